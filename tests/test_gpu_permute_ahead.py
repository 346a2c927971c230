"""Constant defaults of a permute that the scan in front of it fills (Program::prepareAhead): values of every size, defaults longer
and shorter than the scan's share, positions nothing is written to, one scan and two at once, against numpy."""
import numpy as np
import pytest

from accelerate_amd import hip, ir as A

Int = A.Int
TYPES = [(A.i64, np.int64, -3), (A.i32, np.int32, 7), (A.u8, np.uint8, 200), (A.i16, np.int16, -2), (A.f32, np.float32, 0.1),
         (A.f64, np.float64, -0.0)]


def _program(ty, default, two, bound, generate=None):
    """keep the values whose flag is set, in order, over `like`'s extent of defaults; `two`: the others' number as well, by a
    second scan; generate(like, total): other defaults than one constant"""
    V, VI, S0, sh1 = A.tarray(1, ty), A.tarray(1, Int), A.tarray(0, Int), A.tshape(1)
    add = A.lam([Int, Int], lambda x, y: A.add(Int, x, y))

    def scan(of, flags):
        src = A.delayed(VI, A.shape(flags), A.lam([sh1], lambda ix: of(A.index(flags, A.vexp(ix)))),
                        A.lam([Int], lambda i: of(A.linearindex(flags, i))))
        return A.scan_("l", add, A.constI(0), src)

    def body(xs, flags, like):
        def move(places, total):
            to = A.lam([sh1], lambda ix: A.cond(A.eq(Int, A.index(flags, A.vexp(ix)), A.constI(1)),
                                                A.just(A.sh(A.index(places, A.vexp(ix)))), A.nothing(sh1)))
            gen = generate(like, total) if generate else A.generate(V, A.shape(like), A.lam([sh1], lambda ix: A.const(ty, default)))
            return A.permute(A.lam([ty, A.wild(ty)], lambda x, _: x), gen, to, xs)

        def rest(places, total):
            if bound:
                return A.alet(V, move(places, total), lambda r: A.apair(r, total))
            return move(places, total)
        first = lambda k: A.alet(A.tpair(VI, S0), scan(lambda f: f, flags), k)
        if not two:
            return first(lambda a: rest(a[0], a[1]))
        return first(lambda a: A.alet(A.tpair(VI, S0), scan(lambda f: A.sub(Int, A.constI(1), f), flags), lambda b: rest(a[0], b[1])))

    return A.alam([V, VI, VI], body)


@pytest.mark.gpu
@pytest.mark.parametrize("two,bound", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("ty,npty,default", TYPES, ids=[t[0] for t in TYPES])
def test_defaults_filled_by_the_scan(gpu_ctx, knobs, ty, npty, default, two, bound):
    p = gpu_ctx.compile(_program(ty, default, two, bound))
    rng = np.random.default_rng(6)
    for n, m in ((1, 1), (5, 3), (100, 101), (1000, 9001), (2000, 100003), (4097, 4097), (300001, 250007), (1000003, 1000003)):
        x = rng.integers(0, 100, n).astype(npty)
        flags = rng.integers(0, 2, n)
        like = np.zeros(m, np.int64)
        args = [gpu_ctx.to_device(x, A.tarray(1, ty)), gpu_ctx.to_device(flags, A.tarray(1, Int)), gpu_ctx.to_device(like, A.tarray(1, Int))]
        want = np.full(m, default, npty)
        kept = x[flags == 1][:m]
        if int(flags.sum()) > m:
            continue   # (a position outside the destination is an error)
        want[:len(kept)] = kept
        launches = []
        for ahead in (0, 1):
            knobs("permute_ahead", ahead)
            start = gpu_ctx.stat("launches")
            r = p.execute(*args)
            launches.append(gpu_ctx.stat("launches") - start)
            if bound:
                r, total = r.to_host()
                assert total == (n - flags.sum() if two else flags.sum())
            else:
                r = r.to_host()
            assert np.array_equal(r.view(np.uint8), want.view(np.uint8)), (n, m, ahead)
        # (64 KiB a workgroup of the scan: the longest defaults of the short scans stay with their own launch)
        own = m * want.itemsize > 65536 * -(-n // 4096)
        assert own or launches[1] == launches[0] - 1, (n, m, launches)


def _generate(ty, shape, f):
    return A.generate(A.tarray(1, ty), shape, A.lam([A.tshape(1)], f))


# programs that only look alike: (type, defaults, what they are for m of them)
ALIKE = {
    "reads an array": (A.i64, lambda like, total: _generate(A.i64, A.shape(like), lambda ix: A.index(like, A.vexp(ix))), lambda m, t: np.arange(m)),
    "depends on the place": (A.i64, lambda like, total: _generate(A.i64, A.shape(like), lambda ix: A.linearindex(like, A.constI(0))), lambda m, t: np.zeros(m, np.int64)),
    "reads the scan": (A.i64, lambda like, total: _generate(A.i64, A.shape(like), lambda ix: A.index(total, A.nil)), lambda m, t: np.full(m, t)),
    "nan": (A.f32, lambda like, total: _generate(A.f32, A.shape(like), lambda ix: A.const(A.f32, float("nan"))),
            lambda m, t: np.full(m, np.nan, np.float32)),
    "inf": (A.f64, lambda like, total: _generate(A.f64, A.shape(like), lambda ix: A.const(A.f64, float("-inf"))), lambda m, t: np.full(m, -np.inf)),
    "half": (A.f16, lambda like, total: _generate(A.f16, A.shape(like), lambda ix: A.const(A.f16, 1.5)), lambda m, t: np.full(m, 1.5, np.float16)),
}
# the extent is the scan's own total: no launch of the scan can know it
EXTENT = (A.i64, lambda like, total: _generate(A.i64, A.sh(A.index(total, A.nil)), lambda ix: A.const(A.i64, 4)), lambda m, t: np.full(t, 4))


@pytest.mark.parametrize("two", [False, True])
def test_which_scans_fill(capfd, two):
    """the generated source says which scans take a buffer to fill"""
    def fills(program, which=None):
        ctx = hip.Context(-1)
        try:
            ctx.flags = ctx.flags | ctx.FLAG_DUMP_CC
            capfd.readouterr()
            ctx.compile(program)
            return capfd.readouterr().err.count("#define ACC_SCAN_FILL 1")
        finally:
            ctx.close()
    # the scan before the permute, and the pair
    assert fills(_program(A.i64, 0, two, True)) == (2 if two else 1)
    for name, (ty, generate, _) in ALIKE.items():
        assert fills(_program(ty, 0, two, True, generate)) == 0, name
    # nothing follows, or another scan
    V, add = A.tarray(1, Int), A.lam([Int, Int], lambda x, y: A.add(Int, x, y))
    assert fills(A.alam([V], lambda xs: A.alet(V, A.scan("l", add, None, xs), lambda a: A.scan("l", add, None, a)))) == 0


def _run(ctx, knobs, p, args, ahead):
    """results, and how many launches and blocks of memory they took"""
    knobs("permute_ahead", ahead)
    work = lambda: np.array([ctx.stat("launches"), ctx.stat("pool_hits") + ctx.stat("pool_misses")])
    start = work()
    r = p.execute(*args)
    took = work() - start
    r, total = r.to_host()
    return r, total, list(took)


@pytest.mark.gpu
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("name", sorted(ALIKE) + ["extent"])
def test_other_defaults(gpu_ctx, knobs, name, two):
    ty, generate, want_of = EXTENT if name == "extent" else ALIKE[name]
    npty = {A.i64: np.int64, A.f32: np.float32, A.f64: np.float64, A.f16: np.float16}[ty]
    p = gpu_ctx.compile(_program(ty, 0, two, True, generate))
    rng = np.random.default_rng(7)
    for n in (5, 4097, 300001):
        x, flags = rng.integers(0, 100, n).astype(npty), rng.integers(0, 2, n)
        if two:
            flags &= rng.integers(0, 2, n)  # (fewer than the others, whose number may be the extent)
            flags[0] = 0
        t = n - flags.sum() if two else flags.sum()
        args = [gpu_ctx.to_device(x, A.tarray(1, ty)), gpu_ctx.to_device(flags, A.tarray(1, Int)),
                gpu_ctx.to_device(np.arange(n), A.tarray(1, Int))]
        want = want_of(n, t)
        want[:flags.sum()] = x[flags == 1]
        got = [_run(gpu_ctx, knobs, p, args, ahead) for ahead in (0, 1)]
        for r, total, work in got:
            assert total == t and work == got[0][2]
            assert np.array_equal(r.view(np.uint8), want.view(np.uint8)), (n, name)


@pytest.mark.gpu
@pytest.mark.parametrize("two", [False, True])
def test_not_filled_and_not_held(gpu_ctx, knobs, two):
    """defaults of more than 64 KiB a tile, pairs beyond the line, programs that may not work in place: the same launches as without
    it, and no memory taken for defaults that are filled later all the same"""
    p = gpu_ctx.compile(_program(A.i64, -1, two, True))
    rng = np.random.default_rng(8)
    for n, m, inplace in ((5000, 3000000, True), (4200000, 4200000, True), (5000, 5000, False)):
        flags = rng.integers(0, 2, n)
        args = [gpu_ctx.to_device(np.arange(n), A.tarray(1, A.i64)), gpu_ctx.to_device(flags, A.tarray(1, Int)),
                gpu_ctx.to_device(np.zeros(m, np.int64), A.tarray(1, Int))]
        want = np.full(m, -1)
        want[:flags.sum()] = np.arange(n)[flags == 1]
        before = gpu_ctx.flags
        if not inplace:
            gpu_ctx.flags = before & ~gpu_ctx.FLAG_INPLACE
        try:
            got = [_run(gpu_ctx, knobs, p, args, ahead) for ahead in (0, 1)]
        finally:
            gpu_ctx.flags = before
        for r, _, work in got:
            assert work == got[0][2] and np.array_equal(r, want), (n, m)
