"""Loops of stencil sweeps (awhile around a rank-2 stencil of its own state): several iterations
computed in one pass (stencil2d_sweeps.hpp) against the same program with one launch per sweep, which
the oracle tests cover.  A sweep's function fixes the order of its operations, so results are equal
bit for bit."""
import numpy as np
import pytest

from accelerate_amd import ir as A, programs as P

from . import progs as Q

Int = A.Int
BOUNDARIES = ["clamp", "mirror", "wrap", "constant"]
# extents at the edges of the kernel's strips (128 / 256 columns less 2 x 10, 8, 4, 2 margins of 1 or 2) and chunks
SHAPES = [(32, 32), (33, 47), (37, 240), (64, 241), (40, 255), (95, 256), (41, 497), (257, 112), (130, 1003), (1001, 123)]


def _boundary(kind, ty):
    return A.constant(ty, 3) if kind == "constant" else kind


def sweeps(step, ty):
    """the grid after as many sweeps as the second argument, a scalar, says"""
    grid, cnt = A.tarray(2, ty), A.tarray(0, Int)
    state = A.tpair(A.tpair(A.unit, grid), cnt)

    def prog(g0, n):
        loop = A.awhile(state, lambda st: A.unit_(A.u8, A.gt(Int, A.index(st[1], A.nil), A.constI(0))),
                        lambda st: A.apair(A.apair(A.anil, A.apply(step(), st[0][1])),
                                           A.unit_(Int, A.sub(Int, A.index(st[1], A.nil), A.constI(1)))),
                        A.apair(A.apair(A.anil, g0), A.unit_(Int, A.index(n, A.nil))))
        return A.alet(state, loop, lambda st: st[0][1])

    return A.alam([grid, cnt], prog)


def fixed_sweeps(step, ty, count):
    """... as many as a constant says: the loop's counter never needs the device"""
    grid, cnt = A.tarray(2, ty), A.tarray(0, Int)
    state = A.tpair(cnt, grid)

    def prog(g0):
        loop = A.awhile(state, lambda st: A.unit_(A.u8, A.lt(Int, A.index(st[0], A.nil), A.constI(count))),
                        lambda st: A.apair(A.unit_(Int, A.add(Int, A.index(st[0], A.nil), A.constI(1))),
                                           A.apply(step(), st[1])),
                        A.apair(A.unit_(Int, A.constI(0)), g0))
        return A.alet(state, loop, lambda st: st[1])

    return A.alam([grid], prog)


def _grid(shape, npty, seed):
    rng = np.random.default_rng(seed)
    if np.dtype(npty).kind == "f":
        g = rng.uniform(-1, 1, shape).astype(npty)
        g[3, 5], g[-1, -1], g[7, 0] = np.inf if seed == 1 else 1, -0.0, np.finfo(npty).tiny / 4
        return g
    return rng.integers(-1 << 30, 1 << 30, shape).astype(npty)


def _both(ctx, knobs, prog):
    fused = ctx.compile(prog)
    knobs("stencil_sweeps", 0)
    single = ctx.compile(prog)
    knobs("stencil_sweeps", 1)
    assert len(fused.kernel_keys) == len(single.kernel_keys) + 1   # the kernel under test is there
    return fused, single


@pytest.mark.gpu
@pytest.mark.parametrize("kind", BOUNDARIES)
@pytest.mark.parametrize("ty,npty,widths", [
    (A.f32, np.float32, (3, 3)), (A.f32, np.float32, (5, 5)), (A.f32, np.float32, (3, 5)), (A.f32, np.float32, (5, 3)),
    (A.f64, np.float64, (3, 3)), (A.f64, np.float64, (3, 5)), (A.f64, np.float64, (5, 5)), (A.i32, np.int32, (3, 3)), (A.i64, np.int64, (5, 5))], ids=str)
def test_sweeps_equal_single_launches(gpu_ctx, knobs, ty, npty, kind, widths):
    step = lambda: Q.stencil_weighted(ty, widths, _boundary(kind, ty))
    fused, single = _both(gpu_ctx, knobs, sweeps(step, ty))
    for k, shape in enumerate(SHAPES):
        g = gpu_ctx.to_device(_grid(shape, npty, k), A.tarray(2, ty))
        # (integer arithmetic wraps; one grid holds an infinity, and its NaNs compare equal)
        for n in ((1, 2, 3, 7, 8, 13) if k < 3 else (2 + k, 8)):
            cnt = gpu_ctx.to_device(np.array(n, np.int64), A.tarray(0, Int))
            got, want = fused.execute(g, cnt).to_host(), single.execute(g, cnt).to_host()
            assert np.array_equal(got, want, equal_nan=np.dtype(npty).kind == "f"), (shape, n)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", BOUNDARIES)
@pytest.mark.parametrize("ty,npty,taps", [(A.f32, np.float32, "cross"), (A.f64, np.float64, "cross"), (A.i32, np.int32, "row")], ids=str)
def test_neighbours_of_one_row(gpu_ctx, knobs, ty, npty, kind, taps):
    """Functions that tap neighbours in one row only fetch them late and take passes of 10; every number of sweeps up to
    two passes, with results stored past the caches or not."""
    def step():
        sr = A.stup(*[A.sunit(3, ty)] * 3)

        def f(st):
            (_, t, _), (l, c, r), (_, b, _) = (A.untup(row) for row in A.untup(st))
            if taps == "row":
                return A.sub(ty, A.add(ty, l, A.mul(ty, A.const(ty, 3), c)), r)
            return A.sub(ty, A.add(ty, t, A.mul(ty, A.const(ty, 3), l)), A.add(ty, A.add(ty, r, r), b))
        return A.alam([A.tarray(2, ty)], lambda g: A.stencil(sr, ty, A.lam([A.stencil_type(sr)], f), _boundary(kind, ty), g))

    fused, single = _both(gpu_ctx, knobs, sweeps(step, ty))
    for k, (shape, counts) in enumerate([((32, 33), range(1, 12)), ((61, 109), (10, 19)), ((47, 233), (9, 10, 20)),
                                         ((130, 465), (10, 13)), ((300, 240), (3, 7, 10))]):
        g = gpu_ctx.to_device(_grid(shape, npty, 2 + k), A.tarray(2, ty))
        for n in counts:
            cnt = gpu_ctx.to_device(np.array(n, np.int64), A.tarray(0, Int))
            want = single.execute(g, cnt).to_host()
            for stream in (1 << 40, 1):
                knobs("stream_bytes", stream)
                assert np.array_equal(fused.execute(g, cnt).to_host(), want, equal_nan=np.dtype(npty).kind == "f"), (shape, n, stream)


@pytest.mark.gpu
@pytest.mark.parametrize("waves", [2, 64, 100000])
def test_jacobi_by_chunks_of_rows(gpu_ctx, knobs, waves):
    from oracle import c as OC
    fused, _ = _both(gpu_ctx, knobs, fixed_sweeps(P.jacobi_step, A.f32, 19))
    knobs("stencil_sweeps", waves)
    for shape in SHAPES:
        g = np.random.default_rng(5).uniform(0, 1, shape).astype(np.float32)
        got = fused.execute(gpu_ctx.to_device(g, A.tarray(2, A.f32))).to_host()
        assert np.array_equal(got, OC.jacobi_f32(g, 19)), shape


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 1), (1, 40), (31, 64), (64, 31), (0, 64), (64, 0)], ids=str)
def test_extents_below_the_kernels(gpu_ctx, knobs, shape):
    step = lambda: Q.stencil_weighted(A.i32, (3, 3), "clamp")
    fused, single = _both(gpu_ctx, knobs, fixed_sweeps(step, A.i32, 9))
    g = gpu_ctx.to_device(np.arange(shape[0] * shape[1], dtype=np.int32).reshape(shape), A.tarray(2, A.i32))
    assert np.array_equal(fused.execute(g).to_host(), single.execute(g).to_host())


def _state_loop(cond, body):
    grid, cnt = A.tarray(2, A.f32), A.tarray(0, Int)
    state = A.tpair(cnt, grid)
    return A.alam([grid], lambda g0: A.alet(
        state, A.awhile(state, cond, body, A.apair(A.unit_(Int, A.constI(0)), g0)), lambda st: st[1]))


def test_loops_that_read_the_grid_are_left_alone(cc_ctx):
    """No kernel of several sweeps where an iteration's grid is read by anything but the stencil, or
    where the function could not stand lanes outside the array."""
    below = lambda st: A.unit_(A.u8, A.lt(Int, A.index(st[0], A.nil), A.constI(9)))
    up = lambda st: A.unit_(Int, A.add(Int, A.index(st[0], A.nil), A.constI(1)))
    first = lambda g: A.index(g, A.sh(A.constI(0), A.constI(0)))
    plain = lambda st: A.apair(up(st), A.apply(P.jacobi_step(), st[1]))
    extent = lambda st: A.apair(
        A.unit_(Int, A.add(Int, A.shapesize(2, A.shape(st[1])), A.index(st[0], A.nil))), A.apply(P.jacobi_step(), st[1]))
    reads_cond = lambda st: A.unit_(A.u8, A.lt(A.f32, first(st[1]), A.const(A.f32, 9.0)))
    reads_body = lambda st: A.apair(
        A.unit_(Int, A.cond(A.lt(A.f32, first(st[1]), A.const(A.f32, 0.5)), A.constI(9), A.constI(1))),
        A.apply(P.jacobi_step(), st[1]))
    twice = lambda st: A.apair(up(st), A.apply(P.jacobi_step(), A.apply(P.jacobi_step(), st[1])))
    mapped = lambda st: A.apair(up(st), A.map_(A.f32, A.lam([A.f32], lambda v: v), A.apply(P.jacobi_step(), st[1])))
    kept = lambda st: A.apair(up(st), st[1])
    for cond, body, fused in [(below, plain, True), (below, extent, True), (reads_cond, plain, False), (below, reads_body, False),
                              (below, twice, False), (below, mapped, False), (below, kept, False)]:
        prog = _state_loop(cond, body)
        on = cc_ctx.compile(prog).kernel_keys
        old = cc_ctx.set_knob("stencil_sweeps", 0)
        try:
            off = cc_ctx.compile(prog).kernel_keys
        finally:
            cc_ctx.set_knob("stencil_sweeps", old)
        assert len(on) - len(off) == (1 if fused else 0)


def _nine(ty, fn, boundary="clamp"):
    """a step over the nine taps of a 3 x 3 pattern, row by row"""
    row = A.sunit(3, ty)
    sr = A.stup(row, row, row)
    f = A.lam([A.stencil_type(sr)], lambda st: fn([t for r in A.untup(st) for t in A.untup(r)]))
    return A.alam([A.tarray(2, ty)], lambda g: A.stencil(sr, ty, f, boundary, g))


def _kernels(ctx, prog, knob, on):
    """keys of the program with the knob at `on`, and with it off"""
    old = ctx.set_knob(knob, on)
    try:
        with_it = ctx.compile(prog).kernel_keys
        ctx.set_knob(knob, 0)
        return with_it, ctx.compile(prog).kernel_keys
    finally:
        ctx.set_knob(knob, old)


# Lanes in the margins of a strip compute on combinations of values that the array does not hold, so no
# operation of the function may be undefined for any of them (a division by what happens to be zero is, and the compiler
# may drop all that leads there).
_FLOOR = lambda t: A.fromintegral(A.i32, A.f32, A.floor(A.f32, A.i32, t))
PARTIAL = {
    "rem": (A.i32, lambda t: A.rem(A.i32, A.const(A.i32, 1000003), t[4])),
    "quot": (A.i32, lambda t: A.add(A.i32, A.quot(A.i32, t[4], t[5]), t[1])),
    "idiv": (A.i64, lambda t: A.idiv(A.i64, t[4], t[5])),
    "mod": (A.i64, lambda t: A.mod(A.i64, t[4], A.bor(A.i64, t[5], A.const(A.i64, 1)))),
    "quotrem": (A.u32, lambda t: A.let(A.tpair(A.u32, A.u32), A.quotrem(A.u32, t[0], t[8]), lambda v: A.add(A.u32, v[0], v[1]))),
    "divmod": (A.i32, lambda t: A.let(A.tpair(A.i32, A.i32), A.divmod_(A.i32, t[0], t[8]), lambda v: A.add(A.i32, v[0], v[1]))),
    "by zero": (A.i32, lambda t: A.quot(A.i32, t[4], A.const(A.i32, 0))),
    "by minus one": (A.i32, lambda t: A.quot(A.i32, t[4], A.const(A.i32, -1))),
    "guarded": (A.i32, lambda t: A.cond(A.eq(A.i32, t[5], A.const(A.i32, 0)), t[4], A.quot(A.i32, t[4], t[5]))),
    "floor": (A.f32, lambda t: _FLOOR(A.add(A.f32, t[4], t[5]))),
    "rotr": (A.i64, lambda t: A.rotr(A.i64, t[4], t[5])),
    "fromindex": (A.i64, lambda t: A.let(A.tshape(2), A.fromindex(2, A.sh(t[1], t[3]), t[4]), lambda ix: ix[1])),
    "no alternative": (A.i32, lambda t: A.case(A.fromintegral(A.i32, A.u8, t[4]), [(0, t[1]), (1, t[3])])),
}
TOTAL = {
    "by a constant": (A.i32, lambda t: A.add(A.i32, A.quot(A.i32, t[4], A.const(A.i32, 3)), A.mod(A.i32, t[5], A.const(A.i32, 7)))),
    "shifts": (A.i32, lambda t: A.bxor(A.i32, A.shl(A.i32, t[4], A.constI(3)), A.shr(A.i32, t[5], A.fromintegral(A.i32, A.Int, t[3])))),
    "rotates": (A.i64, lambda t: A.bxor(A.i64, A.rotl(A.i64, t[4], t[5]), A.rotr(A.i64, t[3], A.constI(5)))),
    "fdiv": (A.f32, lambda t: A.fdiv(A.f32, t[4], t[5])),
    "alternatives": (A.i32, lambda t: A.case(A.fromintegral(A.i32, A.u8, t[4]), [(0, t[1]), (1, t[3])], t[7])),
}


def test_functions_undefined_for_some_values_are_left_alone(cc_ctx):
    for name, (ty, fn) in list(PARTIAL.items()) + list(TOTAL.items()):
        on, off = _kernels(cc_ctx, fixed_sweeps(lambda: _nine(ty, fn, "wrap"), ty, 9), "stencil_sweeps", 1)
        assert len(on) - len(off) == (1 if name in TOTAL else 0), name


def _window(g, kind):
    """the nine taps of every element"""
    p = np.pad(g, 1, **({"mode": "constant", "constant_values": 3} if kind == "constant" else
                        {"mode": {"clamp": "edge", "mirror": "reflect", "wrap": "wrap"}[kind]}))
    return [p[y:y + g.shape[0], x:x + g.shape[1]] for y in range(3) for x in range(3)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", BOUNDARIES)
def test_division_by_a_tap(gpu_ctx, kind):
    # 2 + 1000003 rem (centre + up): never zero
    step = lambda t: A.add(A.i32, A.const(A.i32, 2), A.rem(A.i32, A.const(A.i32, 1000003), A.add(A.i32, t[4], t[1])))
    run = gpu_ctx.compile(fixed_sweeps(lambda: _nine(A.i32, step, _boundary(kind, A.i32)), A.i32, 5))
    for shape in SHAPES:
        g = np.random.default_rng(2).integers(1, 5000, shape).astype(np.int32)
        want = g
        for _ in range(5):
            w = _window(want, kind)
            want = (2 + 1000003 % (w[4] + w[1])).astype(np.int32)
        assert np.array_equal(run.execute(gpu_ctx.to_device(g, A.tarray(2, A.i32))).to_host(), want), shape


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(TOTAL))
def test_total_functions_equal_single_launches(gpu_ctx, knobs, name):
    ty, fn = TOTAL[name]
    npty = {A.i32: np.int32, A.i64: np.int64, A.f32: np.float32}[ty]
    for kind in BOUNDARIES:
        fused, single = _both(gpu_ctx, knobs, fixed_sweeps(lambda: _nine(ty, fn, _boundary(kind, ty)), ty, 11))
        for k, shape in enumerate(SHAPES):
            g = gpu_ctx.to_device(_grid(shape, npty, k), A.tarray(2, ty))
            got, want = fused.execute(g).to_host(), single.execute(g).to_host()
            assert np.array_equal(got, want, equal_nan=np.dtype(npty).kind == "f"), (kind, shape)


def _sum(ty, widths, boundary):
    """the sum of the taps of a pattern that may be one row, one column or one element"""
    row = A.sunit(widths[1], ty)
    sr = A.stup(*[row] * widths[0])

    def f(st):
        acc = A.const(ty, 1)
        for r in A.untup(st):
            for t in A.untup(r):
                acc = A.add(ty, A.mul(ty, A.const(ty, 0.5 if ty in (A.f32, A.f64) else 3), acc), t)
        return acc

    return A.alam([A.tarray(2, ty)], lambda g: A.stencil(sr, ty, A.lam([A.stencil_type(sr)], f), boundary, g))


FLAT = [(1, 3), (3, 1), (1, 5), (5, 1), (1, 1)]


def test_patterns_of_one_row_or_column_get_the_kernel(cc_ctx):
    for widths in FLAT + [(3, 3), (5, 5), (3, 7), (7, 1)]:
        prog = fixed_sweeps(lambda: _sum(A.i32, widths, "clamp"), A.i32, 9)
        on, off = _kernels(cc_ctx, prog, "stencil_sweeps", 1)
        assert len(on) - len(off) == (1 if max(widths) <= 5 else 0), widths


@pytest.mark.gpu
@pytest.mark.parametrize("kind", BOUNDARIES)
@pytest.mark.parametrize("widths", FLAT, ids=str)
@pytest.mark.parametrize("ty,npty", [(A.f32, np.float32), (A.i64, np.int64)], ids=["f32", "i64"])
def test_patterns_of_one_row_or_column(gpu_ctx, knobs, ty, npty, widths, kind):
    fused, single = _both(gpu_ctx, knobs, sweeps(lambda: _sum(ty, widths, _boundary(kind, ty)), ty))
    for k, shape in enumerate(SHAPES):
        g = gpu_ctx.to_device(_grid(shape, npty, k), A.tarray(2, ty))
        for n in (1, 2, 7, 8, 13) if k < 3 else (8 + k,):
            cnt = gpu_ctx.to_device(np.array(n, np.int64), A.tarray(0, Int))
            got, want = fused.execute(g, cnt).to_host(), single.execute(g, cnt).to_host()
            assert np.array_equal(got, want, equal_nan=np.dtype(npty).kind == "f"), (shape, n)


def _chain(ty, name, n):
    """`n` calls, one of the other's result, after the sum of the nine taps"""
    def fn(t):
        acc = t[0]
        for x in t[1:]:
            acc = A.add(ty, acc, x)
        for k in range(n):
            acc = A.prim(name, ty, A.pair(acc, t[k]) if name in ("fpow", "atan2") else acc)
        return acc
    return fn


def test_heavy_functions_are_left_alone(cc_ctx):
    for ty in (A.f32, A.f64):
        for fn, kernel in [(_chain(ty, "abs", 16), True), (_chain(ty, "exp", 1), True), (_chain(ty, "sqrt", 2), True), (_chain(ty, "exp", 4), False),
                           (_chain(ty, "fpow", 1), False), (_chain(ty, "sin", 1), False), (_chain(ty, "recip", 7), False)]:
            on, off = _kernels(cc_ctx, fixed_sweeps(lambda: _nine(ty, fn), ty, 9), "stencil_sweeps", 1)
            assert len(on) - len(off) == (1 if kernel else 0)
    # equal subterms count once
    fn = lambda t: A.add(A.f32, *[A.mul(A.f32, *[_chain(A.f32, "exp", 1)(t)] * 2)] * 2)
    on, off = _kernels(cc_ctx, fixed_sweeps(lambda: _nine(A.f32, fn), A.f32, 9), "stencil_sweeps", 1)
    assert len(on) == len(off) + 1


@pytest.mark.gpu
@pytest.mark.parametrize("kind", BOUNDARIES)
@pytest.mark.parametrize("ty,npty", [(A.f32, np.float32), (A.i64, np.int64)], ids=["f32", "i64"])
def test_functions_of_25_taps_on_small_arrays(gpu_ctx, knobs, ty, npty, kind):
    # one launch a sweep on arrays of this size; a number of waves asks for the kernel all the same
    step = lambda: Q.stencil_weighted(ty, (5, 5), _boundary(kind, ty))
    fused, single = _both(gpu_ctx, knobs, fixed_sweeps(step, ty, 13))
    for k, shape in enumerate(SHAPES):
        g = gpu_ctx.to_device(_grid(shape, npty, k), A.tarray(2, ty))
        want = single.execute(g).to_host()
        for waves, launches in [(1, 13), (3072, 4)]:          # 4 + 4 + 4 + 1
            knobs("stencil_sweeps", waves)
            before = gpu_ctx.stat("launches")
            got = fused.execute(g).to_host()
            assert gpu_ctx.stat("launches") - before == launches
            assert np.array_equal(got, want, equal_nan=np.dtype(npty).kind == "f"), (shape, waves)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,launches", [(5000, 9), (5040, 3)])
def test_functions_of_25_taps_on_large_arrays(gpu_ctx, knobs, rows, launches):
    # 96 MiB are 5033.2 rows of 5000 Float32
    fused, single = _both(gpu_ctx, knobs, fixed_sweeps(lambda: Q.stencil_weighted(A.f32, (5, 5), A.clamp), A.f32, 9))
    g = gpu_ctx.to_device(np.random.default_rng(8).uniform(-1, 1, (rows, 5000)).astype(np.float32), A.tarray(2, A.f32))
    before = gpu_ctx.stat("launches")
    got = fused.execute(g)
    assert gpu_ctx.stat("launches") - before == launches
    assert np.array_equal(got.to_host(), single.execute(g).to_host())
