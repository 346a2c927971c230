"""The scans whose tiles all run at once and each read the aggregates of all their predecessors
(acc_scan_all: 64 bytes a lane, acc_scan_all2: 128), forced through the `scan_tiles` knob onto
lengths at the edges of their tiles, of a wave's and a workgroup's share of predecessors (64, 256) and of
rows, against numpy (Interpreter.hs:427-582)."""
import numpy as np
import pytest

from accelerate_amd import ir as A, programs as P

from . import progs as Q

pytestmark = pytest.mark.gpu

TILES = [1, 2, 3, 64, 65, 66, 256, 257, 300, 512, 514]   # the last tile has 63, 64, 65 .. predecessors


def _lengths(tile):
    out = [1, tile - 1]
    for k in TILES:
        out += [k * tile, k * tile - tile // 2 - 3, (k - 1) * tile + 1]
    return sorted({n for n in out if n > 0})


def _running(x, right):
    y = x[..., ::-1] if right else x
    s = np.cumsum(y, axis=-1, dtype=x.dtype)
    return s[..., ::-1] if right else s


@pytest.mark.parametrize("which", [5, 6])
@pytest.mark.parametrize("d", ["l", "r"])
@pytest.mark.parametrize("ty,npty,size", [(A.i32, np.int32, 4), (A.i64, np.int64, 8), (A.f64, np.float64, 8)],
                         ids=["i32", "i64", "f64"])
def test_every_kind(gpu_ctx, knobs, ty, npty, size, d, which):
    tile = 256 * 64 // size * (which - 4)
    one, seeded, prime = (gpu_ctx.compile(p) for p in (P.scan1_sum(d, ty), P.scan_sum(d, ty, 1, 5), P.scan_prime_sum(d, ty, 1, 3)))
    knobs("scan_tiles", which)
    rng = np.random.default_rng(11)
    for n in _lengths(tile):
        x = rng.integers(-1000, 1000, n).astype(npty)   # (sums of whole numbers: exact in Double too)
        inc = _running(x, d == "r")
        dx = gpu_ctx.to_device(x, A.tarray(1, ty))
        assert np.array_equal(one.execute(dx).to_host(), inc), n
        with_seed = np.concatenate([inc, [0]]) if d == "r" else np.concatenate([[0], inc])
        assert np.array_equal(seeded.execute(dx).to_host(), (5 + with_seed).astype(npty)), n
        body, total = [p.to_host() for p in prime.execute(dx).parts()]
        assert np.array_equal(body, (3 + (with_seed[1:] if d == "r" else with_seed[:-1])).astype(npty)), n
        assert total == 3 + inc[0 if d == "r" else -1], n


@pytest.mark.parametrize("which", [0, 5, 6])
def test_rows_and_an_operator_that_does_not_commute(gpu_ctx, knobs, which):
    # the last value that is not zero so far: every row starts anew, and order matters
    last = A.lam([A.i64, A.i64], lambda p, q: A.cond(A.neq(A.i64, q, A.constI(0)), q, p))
    run = gpu_ctx.compile(A.alam([A.tarray(2, A.i64)], lambda xs: A.scan("l", last, None, xs)))
    knobs("scan_tiles", which)
    rng = np.random.default_rng(3)
    for rows, n in [(1, 70 * 2048 + 5), (2, 16385), (3, 40000), (7, 66 * 2048 + 1), (1, 520 * 4096 - 7)]:
        x = rng.integers(1, 1 << 40, (rows, n)) * (rng.random((rows, n)) < 0.0005)
        at = np.maximum.accumulate(np.where(x != 0, np.arange(n), 0), axis=1)
        want = np.take_along_axis(x, at, 1)
        assert np.array_equal(run.execute(gpu_ctx.to_device(x, A.tarray(2, A.i64))).to_host(), want), (rows, n)


def test_wide_elements(gpu_ctx, knobs):
    # pairs: descriptors of three words
    ty = A.ttup(A.i32, A.i64)
    add = A.lam([ty, ty], lambda x, y: A.tup(A.add(A.i32, A.untup(x)[0], A.untup(y)[0]), A.add(A.i64, A.untup(x)[1], A.untup(y)[1])))
    run = gpu_ctx.compile(A.alam([A.tarray(1, A.i32), A.tarray(1, A.i64)], lambda a, b: A.scan(
        "l", add, None, A.zipwith(ty, A.lam([A.i32, A.i64], lambda p, q: A.tup(p, q)), a, b))))
    rng = np.random.default_rng(4)
    for which in (5, 6):
        knobs("scan_tiles", which)
        for n in (1000, 100001, 700001):
            a, b = rng.integers(-99, 99, n).astype(np.int32), rng.integers(-1 << 40, 1 << 40, n)
            got = run.execute(gpu_ctx.to_device(a, A.tarray(1, A.i32)), gpu_ctx.to_device(b, A.tarray(1, A.i64))).to_host()
            for g, w in zip(got, (np.cumsum(a, dtype=np.int32), np.cumsum(b))):
                assert np.array_equal(np.asarray(g), w), (which, n)


@pytest.mark.parametrize("which", [5, 6])
@pytest.mark.parametrize("d", ["l", "r"])
@pytest.mark.parametrize("ty,npty,size", [(A.i32, np.int32, 4), (A.i64, np.int64, 8)], ids=["i32", "i64"])
def test_every_kind_over_rows(gpu_ctx, knobs, ty, npty, size, d, which):
    # a tile belongs to one row; rows that end in, just before and just after a tile's last value
    tile = 256 * 64 // size * (which - 4)
    progs = [gpu_ctx.compile(p) for p in (P.scan1_sum(d, ty, 2), P.scan_sum(d, ty, 2, 5), P.scan_prime_sum(d, ty, 2, 3))]
    knobs("scan_tiles", which)
    rng = np.random.default_rng(12)
    for rows, n in [(2, tile // 2 + 3), (5, tile - 1), (3, tile), (4, tile + 1), (7, 2 * tile + 5), (2, 65 * tile + 1), (3, 66 * tile - 3)]:
        x = rng.integers(-1000, 1000, (rows, n)).astype(npty)
        inc = _running(x, d == "r")
        none = np.zeros((rows, 1), npty)
        with_seed = np.concatenate([inc, none] if d == "r" else [none, inc], axis=1)
        dx = gpu_ctx.to_device(x, A.tarray(2, ty))
        assert np.array_equal(progs[0].execute(dx).to_host(), inc), (rows, n)
        assert np.array_equal(progs[1].execute(dx).to_host(), 5 + with_seed), (rows, n)
        body, total = [p.to_host() for p in progs[2].execute(dx).parts()]
        assert np.array_equal(body, 3 + (with_seed[:, 1:] if d == "r" else with_seed[:, :-1])), (rows, n)
        assert np.array_equal(total, 3 + inc[:, 0 if d == "r" else -1]), (rows, n)
