"""Constant defaults of a permute that the scan in front of it fills (Program::prepareAhead): values of every size, defaults longer
and shorter than the scan's share, positions nothing is written to, one scan and two at once, against numpy."""
import numpy as np
import pytest

from accelerate_amd import ir as A

Int = A.Int
TYPES = [(A.i64, np.int64, -3), (A.i32, np.int32, 7), (A.u8, np.uint8, 200), (A.i16, np.int16, -2), (A.f32, np.float32, 0.1),
         (A.f64, np.float64, -0.0)]


def _program(ty, default, two, bound):
    """keep the values whose flag is set, in order, over `like`'s extent of defaults; `two`: the others' number as well, by a
    second scan"""
    V, VI, S0, sh1 = A.tarray(1, ty), A.tarray(1, Int), A.tarray(0, Int), A.tshape(1)
    add = A.lam([Int, Int], lambda x, y: A.add(Int, x, y))

    def scan(of, flags):
        src = A.delayed(VI, A.shape(flags), A.lam([sh1], lambda ix: of(A.index(flags, A.vexp(ix)))),
                        A.lam([Int], lambda i: of(A.linearindex(flags, i))))
        return A.scan_("l", add, A.constI(0), src)

    def body(xs, flags, like):
        def move(places):
            to = A.lam([sh1], lambda ix: A.cond(A.eq(Int, A.index(flags, A.vexp(ix)), A.constI(1)),
                                                A.just(A.sh(A.index(places, A.vexp(ix)))), A.nothing(sh1)))
            return A.permute(A.lam([ty, A.wild(ty)], lambda x, _: x),
                             A.generate(V, A.shape(like), A.lam([sh1], lambda ix: A.const(ty, default))), to, xs)

        def rest(places, total):
            if bound:
                return A.alet(V, move(places), lambda r: A.apair(r, total))
            return move(places)
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


def test_scan_and_what_follows(cc_ctx):
    # (programs that only look alike are compiled all the same: the defaults read an array, or are no constant)
    for two in (False, True):
        assert cc_ctx.compile(_program(A.i64, 0, two, True)).num_kernels > 0
