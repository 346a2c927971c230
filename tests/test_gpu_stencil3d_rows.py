"""Rank-3 stencils of many taps computed from registers (stencil3d_rows.hpp) against the kernel that goes
through LDS, which the oracle tests cover: the function fixes the order of its operations, so results
are equal bit for bit."""
import numpy as np
import pytest

from accelerate_amd import ir as A

pytestmark = pytest.mark.gpu

# extents at the edges of a strip (124 columns of the 128 its lanes hold), of the four bands of 4 or 2 rows of a
# workgroup and of the loop's three planes; the smallest
SHAPES = [(2, 2, 2), (3, 3, 5), (1, 4, 7), (5, 1, 64), (4, 9, 123), (6, 8, 124), (7, 31, 125), (9, 16, 128), (3, 5, 249),
          (33, 17, 126), (12, 100, 130), (5, 33, 248)]


def _backward(ty, nx, out, boundary):
    """all taps of 3 x 3 x nx from the last plane to the first, distinct weights: no function to be taken plane by plane"""
    row = A.sunit(nx, ty)
    sr = A.stup(*[A.stup(row, row, row)] * 3)

    def f(st):
        ts = [t for p in A.untup(st) for r in A.untup(p) for t in A.untup(r)]
        acc = A.const(out, 1)
        for k, t in enumerate(reversed(ts)):
            t = t if ty == out else A.fromintegral(ty, out, t)
            acc = A.add(out, acc, A.mul(out, A.const(out, k + 1), t))
        return acc

    return A.alam([A.tarray(3, ty)], lambda g: A.stencil(sr, out, A.lam([A.stencil_type(sr)], f), boundary, g))


def _launched(ctx, capfd, prog, arg):
    """the result, and the names of what was launched"""
    before = ctx.flags
    ctx.flags = before | ctx.FLAG_DUMP_EXEC
    capfd.readouterr()
    try:
        out = prog.execute(arg)
    finally:
        ctx.flags = before
    return out, capfd.readouterr().err


@pytest.mark.parametrize("chain", [0, 7])
@pytest.mark.parametrize("kind", ["clamp", "mirror", "wrap", "constant"])
@pytest.mark.parametrize("ty,npty,nx", [(A.f32, np.float32, 3), (A.f64, np.float64, 3), (A.i32, np.int32, 3), (A.i64, np.int64, 3),
                                        (A.i32, np.int32, 1)], ids=str)
def test_equal_to_the_lds_kernel(gpu_ctx, knobs, capfd, ty, npty, nx, kind, chain):
    # (of 3 x 3 x 1 taps to a result of another type)
    prog = _backward(ty, nx, ty if nx > 1 else A.i64, A.constant(ty, 3) if kind == "constant" else kind)
    knobs("stencil_rows3d", 0)
    lds = gpu_ctx.compile(prog)
    knobs("stencil_rows3d", 2)
    rows = gpu_ctx.compile(prog)
    assert lds.kernel_keys != rows.kernel_keys
    rng = np.random.default_rng(6)
    for shape in SHAPES:
        if kind == "mirror" and min(shape[:2] + (shape[2:] if nx > 1 else ())) < 2:
            continue  # refused: shorter than the taps reach
        g = rng.integers(-999, 999, shape).astype(npty)
        if np.dtype(npty).kind == "f":
            g *= npty(0.37)
        d = gpu_ctx.to_device(g, A.tarray(3, ty))
        want = lds.execute(d).to_host()
        knobs("stencil_chain", chain)
        got, names = _launched(gpu_ctx, capfd, rows, d)
        knobs("stencil_chain", 0)
        assert "acc_stencil3d_rows" in names, shape
        assert np.array_equal(got.to_host(), want), shape


# Both kernels are compiled; a launch takes the one that is faster on its extents.  Below 192 MiB of operand and
# result from registers; up to 512 MiB (of 4-byte elements) where strips of 124 columns are filled to 0.7 of 128; beyond, where tiles of 128
# columns are filled to less than 0.8.
@pytest.mark.parametrize("shape,taps,rows", [
    ((6, 8, 124), 27, True), ((200, 200, 200), 19, True), ((290, 295, 300), 19, False), ((290, 295, 300), 27, True),
    ((500, 256, 256), 27, False), ((512, 512, 512), 27, False), ((640, 400, 300), 27, True)], ids=str)
def test_the_kernel_a_launch_takes(gpu_ctx, knobs, capfd, shape, taps, rows):
    row = A.sunit(3, A.f32)
    sr = A.stup(*[A.stup(row, row, row)] * 3)

    def f(st):
        ts = [t for p in A.untup(st) for r in A.untup(p) for t in A.untup(r)]
        acc = ts[13]
        for k, t in enumerate(ts[:taps - 1]):
            acc = A.add(A.f32, acc, A.mul(A.f32, A.const(A.f32, 0.01 * (k + 1)), t))
        return acc if taps < 27 else A.add(A.f32, acc, ts[26])

    prog = gpu_ctx.compile(A.alam([A.tarray(3, A.f32)], lambda g: A.stencil(sr, A.f32, A.lam([A.stencil_type(sr)], f), A.clamp, g)))
    g = gpu_ctx.to_device(np.random.default_rng(9).random(shape, dtype=np.float32), A.tarray(3, A.f32))
    got = {}
    for knob in (1, 0, 2):
        knobs("stencil_rows3d", knob)
        out, names = _launched(gpu_ctx, capfd, prog, g)
        assert ("acc_stencil3d_rows" in names) == (knob == 2 or knob == 1 and rows)
        got[knob] = out.to_host()
    assert np.array_equal(got[0], got[2]) and np.array_equal(got[0], got[1])


# plane by plane (stencil3d_planes.hpp): extents at the edges of a lane's columns (4, 2 of 8 bytes, 2 under wrap), of a wave's 62 lanes, of bands of
# three rows and of chunks; the taps a function reads, from one plane or all of them
@pytest.mark.parametrize("kind", ["clamp", "mirror", "wrap", "constant"])
@pytest.mark.parametrize("ty,npty,taps", [(A.f32, np.float32, "all"), (A.f64, np.float64, "cross"), (A.i32, np.int32, "cross"),
                                          (A.i64, np.int64, "ends"), (A.f32, np.float32, "middle")], ids=str)
def test_plane_by_plane(gpu_ctx, knobs, capfd, ty, npty, taps, kind):
    row = A.sunit(3, ty)
    sr = A.stup(*[A.stup(row, row, row)] * 3)
    read = {"all": range(27), "cross": (4, 10, 12, 13, 14, 16, 22), "ends": (0, 26), "middle": (9, 13, 17)}[taps]

    def f(st):
        ts = [t for p in A.untup(st) for r in A.untup(p) for t in A.untup(r)]
        acc = None
        for k in read:
            v = A.mul(ty, A.const(ty, k + 1), ts[k])
            acc = v if acc is None else A.sub(ty, acc, v)
        return acc

    prog = A.alam([A.tarray(3, ty)], lambda g: A.stencil(sr, ty, A.lam([A.stencil_type(sr)], f),
                                                         A.constant(ty, 3) if kind == "constant" else kind, g))
    knobs("stencil_rows3d", 0)
    lds = gpu_ctx.compile(prog)
    knobs("stencil_rows3d", 2)
    planes = gpu_ctx.compile(prog)
    assert lds.kernel_keys != planes.kernel_keys
    rng = np.random.default_rng(8)
    for shape in [(2, 2, 2), (1, 1, 4), (2, 3, 3), (3, 2, 5), (6, 3, 123), (7, 4, 124), (13, 5, 125), (5, 64, 61), (12, 7, 248), (4, 10, 249),
                  (30, 40, 50), (19, 100, 31), (3, 301, 6), (100, 33, 130)]:
        if kind == "mirror" and min(shape) < 2:
            continue  # refused: shorter than the taps reach
        g = rng.integers(-999, 999, shape).astype(npty)
        if np.dtype(npty).kind == "f":
            g *= npty(0.37)
            g[-1, -1, -1], g[0, 0, 0] = np.inf, npty(-0.0)
        d = gpu_ctx.to_device(g, A.tarray(3, ty))
        want = lds.execute(d).to_host()
        for chain in (0, 1, 2, 3, 5):
            knobs("stencil_chain", chain)
            got, names = _launched(gpu_ctx, capfd, planes, d)
            # (rows shorter than a lane's columns go through LDS)
            assert ("acc_stencil3d_planes" in names) == (shape[2] >= (8 if kind == "wrap" else 16) // np.dtype(npty).itemsize), shape
            assert np.array_equal(got.to_host(), want, equal_nan=np.dtype(npty).kind == "f"), (shape, chain)
        knobs("stencil_chain", 0)


@pytest.mark.parametrize("kind", ["clamp", "wrap"])
@pytest.mark.parametrize("out,npout", [(A.u8, np.uint8), (A.i8, np.int8), (A.i16, np.int16), (A.u16, np.uint16)], ids=str)
def test_plane_by_plane_to_small_results(gpu_ctx, knobs, capfd, out, npout, kind):
    row = A.sunit(3, A.i32)
    sr = A.stup(*[A.stup(row, row, row)] * 3)

    def f(st):
        ts = [t for p in A.untup(st) for r in A.untup(p) for t in A.untup(r)]
        acc = ts[0]
        for k in (4, 12, 13, 14, 22, 26):
            acc = A.add(A.i32, acc, A.mul(A.i32, A.const(A.i32, k), ts[k]))
        return A.fromintegral(A.i32, out, acc)

    prog = A.alam([A.tarray(3, A.i32)], lambda g: A.stencil(sr, out, A.lam([A.stencil_type(sr)], f), kind, g))
    knobs("stencil_rows3d", 0)
    lds = gpu_ctx.compile(prog)
    knobs("stencil_rows3d", 2)
    planes = gpu_ctx.compile(prog)
    rng = np.random.default_rng(3)
    for shape in [(1, 1, 4), (3, 2, 5), (5, 4, 7), (2, 64, 61), (7, 7, 125), (4, 10, 249)]:
        d = gpu_ctx.to_device(rng.integers(-9999, 9999, shape).astype(np.int32), A.tarray(3, A.i32))
        got, names = _launched(gpu_ctx, capfd, planes, d)
        assert "acc_stencil3d_planes" in names
        knobs("stencil_rows3d", 0)
        want = lds.execute(d).to_host()
        knobs("stencil_rows3d", 2)
        assert got.to_host().dtype == npout and np.array_equal(got.to_host(), want), shape
