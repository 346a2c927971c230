"""Two scans in a row that do not depend on one another, computed by one launch (Program::evalJoint): every kind and
direction against numpy, one after the other where extents differ, and the pairs that must stay apart."""
import numpy as np
import pytest

from accelerate_amd import ir as A

KINDS = ["scan1", "scan", "scan'"]


def _two(kind, d, t1, t2, rank=1, second=None):
    """(scan (+) xs, scan max (map (* 3) ys)), both let-bound; `second` replaces the second operand by a function of
    what the first scan gave"""
    sh = A.tshape(rank)
    v1, v2 = A.tarray(rank, t1), A.tarray(rank, t2)
    add = A.lam([t1, t1], lambda x, y: A.add(t1, x, y))
    most = A.lam([t2, t2], lambda x, y: A.max_(t2, x, y))

    def scan(f, ty, z, src):
        if kind == "scan'":
            return A.scan_(d, f, A.const(ty, z), src)
        return A.scan(d, f, None if kind == "scan1" else A.const(ty, z), src)

    def bound(v, ty):
        return A.tpair(v, A.tarray(rank - 1, ty)) if kind == "scan'" else v

    def out(r):
        return A.apair(r[0], r[1]) if kind == "scan'" else r

    def body(xs, ys):
        def triple(of):
            f = lambda e: A.mul(t2, A.const(t2, 3), e)
            return A.delayed(v2, A.shape(of), A.lam([sh], lambda ix: f(A.index(of, A.vexp(ix)))),
                             A.lam([A.Int], lambda i: f(A.linearindex(of, i))))
        return A.alet(bound(v1, t1), scan(add, t1, 5, xs), lambda r1: A.alet(
            bound(v2, t2), scan(most, t2, -7, triple(second(r1) if second else ys)), lambda r2: A.apair(out(r1), out(r2))))

    return A.alam([v1, v2], body)


def _numpy(kind, d, f, z, x):
    y = x[..., ::-1] if d == "r" else x
    if kind == "scan1":
        s = f.accumulate(y, axis=-1, dtype=x.dtype)
        return [s[..., ::-1] if d == "r" else s]
    y = np.concatenate([np.full(y.shape[:-1] + (1,), z, x.dtype), y], axis=-1)
    s = f.accumulate(y, axis=-1, dtype=x.dtype)
    if kind == "scan":
        return [s[..., ::-1] if d == "r" else s]
    return [s[..., :-1][..., ::-1] if d == "r" else s[..., :-1], s[..., -1]]


def _leaves(r):
    flat = lambda v: [x for p in v for x in flat(p)] if isinstance(v, tuple) else [v]
    return flat(r.to_host())


TYPES = [(A.i64, np.int64, A.i64, np.int64), (A.i32, np.int32, A.i64, np.int64), (A.f32, np.float32, A.i32, np.int32),
         (A.f64, np.float64, A.u8, np.uint8)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("d", ["l", "r"])
@pytest.mark.parametrize("t1,n1,t2,n2", TYPES, ids=["i64-i64", "i32-i64", "f32-i32", "f64-u8"])
def test_both_at_once(gpu_ctx, knobs, kind, d, t1, n1, t2, n2):
    prog = _two(kind, d, t1, t2)
    p = gpu_ctx.compile(prog)
    rng = np.random.default_rng(4)
    z2 = np.array(-7).astype(n2)
    # around the tiles of every variant (512 .. 8192 elements), and beyond what runs at once
    for n in (1, 2, 255, 511, 513, 1024, 2047, 4097, 8192, 70001, 262144, 1000003):
        # (sums of whole numbers below 2^24: exact in Float32 too)
        x, y = rng.integers(-8, 9, n).astype(n1), rng.integers(0, 80, n).astype(n2)
        args = [gpu_ctx.to_device(x, A.tarray(1, t1)), gpu_ctx.to_device(y, A.tarray(1, t2))]
        start = gpu_ctx.stat("launches")
        got = _leaves(p.execute(*args))
        assert gpu_ctx.stat("launches") == start + 1
        want = _numpy(kind, d, np.add, 5, x) + _numpy(kind, d, np.maximum, z2, y * np.array(3, n2))
        assert len(got) == len(want)
        for g, w in zip(got, want):
            assert np.array_equal(g, w), n


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("tiles", [0, 1, 2, 3, 5, 6])
def test_rows_and_every_variant(gpu_ctx, knobs, kind, tiles):
    p = gpu_ctx.compile(_two(kind, "r" if tiles & 1 else "l", A.i64, A.i32, rank=2))
    knobs("scan_tiles", tiles)
    rng = np.random.default_rng(tiles)
    for shape in ((1, 3000), (3, 1), (700, 7), (5, 400), (2, 20011)) + (() if tiles == 3 else ((3, 70000),)):
        x, y = rng.integers(-1 << 40, 1 << 40, shape), rng.integers(-1 << 20, 1 << 20, shape).astype(np.int32)
        got = _leaves(p.execute(gpu_ctx.to_device(x, A.tarray(2, A.i64)), gpu_ctx.to_device(y, A.tarray(2, A.i32))))
        d = "r" if tiles & 1 else "l"
        want = _numpy(kind, d, np.add, 5, x) + _numpy(kind, d, np.maximum, -7, y * np.int32(3))
        for g, w in zip(got, want):
            assert np.array_equal(g, w), shape


@pytest.mark.gpu
def test_extents_that_differ(gpu_ctx):
    p = gpu_ctx.compile(_two("scan'", "l", A.i64, A.i64))
    for n, m in ((100, 99), (0, 5), (5, 0), (0, 0), (3000, 4001)):
        x, y = np.arange(n), np.arange(m) % 13
        got = _leaves(p.execute(gpu_ctx.to_device(x, A.tarray(1, A.i64)), gpu_ctx.to_device(y, A.tarray(1, A.i64))))
        want = _numpy("scan'", "l", np.add, 5, x) + _numpy("scan'", "l", np.maximum, -7, y * 3)
        for g, w in zip(got, want):
            assert np.array_equal(g, w), (n, m)


@pytest.mark.gpu
@pytest.mark.parametrize("t1,n1,t2,n2,tile", [(A.i64, np.int64, A.i64, np.int64, 4096), (A.f32, np.float32, A.i32, np.int32, 8192),
                                              (A.u8, np.uint8, A.u8, np.uint8, 16384), (A.u8, np.uint8, A.i32, np.int32, 8192),
                                              (A.i16, np.int16, A.i64, np.int64, 4096)], ids=["i64-i64", "f32-i32", "u8-u8", "u8-i32", "i16-i64"])
def test_the_line(gpu_ctx, t1, n1, t2, n2, tile):
    """up to 1024 tiles of what a lane holds of the pairs (a leaf takes four bytes, an element its alignment) in one launch"""
    p = gpu_ctx.compile(_two("scan", "l", t1, t2))
    rng = np.random.default_rng(11)
    for n, launches in ((1024 * tile, 1), (1024 * tile + 1, 2), (700 * tile + 1, 1)):
        x, y = rng.integers(0, 2, n).astype(n1), rng.integers(0, 80, n).astype(n2)
        args = [gpu_ctx.to_device(x, A.tarray(1, t1)), gpu_ctx.to_device(y, A.tarray(1, t2))]
        start = gpu_ctx.stat("launches")
        got = _leaves(p.execute(*args))
        assert gpu_ctx.stat("launches") == start + launches
        want = _numpy("scan", "l", np.add, 5, x) + _numpy("scan", "l", np.maximum, np.array(-7).astype(n2), y * np.array(3, n2))
        for g, w in zip(got, want):
            assert np.array_equal(g, w), n


@pytest.mark.gpu
def test_three_in_a_row_and_in_a_loop(gpu_ctx):
    """three scans share a launch two by two; a pair inside a loop reads each iteration's state"""
    V, Int = A.tarray(1, A.i64), A.Int
    add = A.lam([A.i64, A.i64], lambda x, y: A.add(A.i64, x, y))
    most = A.lam([A.i64, A.i64], lambda x, y: A.max_(A.i64, x, y))
    scan = lambda f, xs: A.scan("l", f, None, xs)
    three = gpu_ctx.compile(A.alam([V, V, V], lambda a, b, c: A.alet(V, scan(add, a), lambda x: A.alet(
        V, scan(most, b), lambda y: A.alet(V, scan(add, c), lambda z: A.apair(x, A.apair(y, z)))))))
    state = A.tpair(A.tpair(V, V), A.tarray(0, Int))
    loop = gpu_ctx.compile(A.alam([V, V], lambda a, b: A.awhile(
        state, lambda st: A.unit_(A.u8, A.lt(Int, A.index(st[1], A.nil), A.constI(3))),
        lambda st: A.alet(V, scan(add, st[0][0]), lambda x: A.alet(V, scan(most, st[0][1]), lambda y: A.apair(
            A.apair(y, x), A.unit_(Int, A.add(Int, A.index(st[1], A.nil), A.constI(1)))))),
        A.apair(A.apair(a, b), A.unit_(Int, A.constI(0))))))
    rng = np.random.default_rng(12)
    for n in (3, 5000, 300001):
        host = [rng.integers(-100, 100, n) for _ in range(3)]
        dev = [gpu_ctx.to_device(x, V) for x in host]
        start = gpu_ctx.stat("launches")
        got = _leaves(three.execute(*dev))
        assert gpu_ctx.stat("launches") == start + 2
        for g, w in zip(got, (np.cumsum(host[0]), np.maximum.accumulate(host[1]), np.cumsum(host[2]))):
            assert np.array_equal(g, w), n
        a, b = host[:2]
        for _ in range(3):
            a, b = np.maximum.accumulate(b), np.cumsum(a)
        start = gpu_ctx.stat("launches")
        x, y, _ = _leaves(loop.execute(*dev[:2]))
        assert gpu_ctx.stat("launches") == start + 3
        assert np.array_equal(x, a) and np.array_equal(y, b), n


def test_which_pairs_are_computed_together(cc_ctx):
    def kernels(prog):
        return len(cc_ctx.compile(prog).kernel_keys)

    def apart(prog):
        old = cc_ctx.set_knob("scan_joint", 0)
        try:
            return kernels(prog)
        finally:
            cc_ctx.set_knob("scan_joint", old)

    together = _two("scan", "l", A.i64, A.i64)
    assert kernels(together) == apart(together) + 1
    # the second reads the first's result
    for prog in (_two("scan1", "l", A.i64, A.i64, second=lambda r: r), _two("scan'", "r", A.i64, A.i64, second=lambda r: r[0])):
        assert kernels(prog) == apart(prog)
    # two directions, or only one of the two with a seed
    V = A.tarray(1, A.i64)
    add = A.lam([A.i64, A.i64], lambda x, y: A.add(A.i64, x, y))
    for one, other in ((("l", None), ("r", None)), (("l", 0), ("l", None)), (("r", None), ("r", 0))):
        scan = lambda k, xs: A.scan(k[0], add, None if k[1] is None else A.const(A.i64, k[1]), xs)
        prog = A.alam([V, V], lambda a, b: A.alet(V, scan(one, a), lambda x: A.alet(V, scan(other, b), lambda y: A.apair(x, y))))
        assert kernels(prog) == apart(prog)
