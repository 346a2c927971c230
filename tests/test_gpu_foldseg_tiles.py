"""Segmented folds over fused producers (Interpreter.hs:390-425): a launch takes tiles of 8192 or 4096 Int32 values by the
number of values, whether the last tile is full, and whether the producer reads an array."""
import re

import numpy as np
import pytest

from accelerate_amd import ir as A

pytestmark = pytest.mark.gpu

Int = A.Int


def _add(ty):
    return A.lam([ty, ty], lambda x, y: A.add(ty, x, y))


def _program(fn):
    """foldSeg (+) 0 (map fn xs) seg"""
    def prog(xs, seg):
        src = A.delayed(A.tarray(1, A.i32), A.shape(xs), A.lam([A.tshape(1)], lambda ix: fn(lambda: A.index(xs, A.vexp(ix)))),
                        A.lam([Int], lambda i: fn(lambda: A.linearindex(xs, A.vexp(i)))))
        return A.alet(A.tarray(1, Int), A.scan("l", _add(Int), A.const(Int, 0), seg),
                      lambda offs: A.foldseg(Int, _add(A.i32), A.const(A.i32, 0), src, offs))
    return A.alam([A.tarray(1, A.i32), A.tarray(1, Int)], prog)


@pytest.mark.parametrize("reads", [True, False], ids=["reads", "constant"])
def test_tiles_of_a_launch(gpu_ctx, capfd, reads):
    fn = (lambda x: A.add(A.i32, A.mul(A.i32, x(), A.const(A.i32, 3)), A.const(A.i32, 1))) if reads else lambda x: A.const(A.i32, 2)
    run = gpu_ctx.compile(_program(fn))
    for n, half in [(1, True), (4095, True), (4097, True), (100003, True), (1 << 22, True), (1 << 23, False), ((1 << 23) + 1, True),
                    ((3 << 23) - 5, True), (3 << 23, False), ((3 << 23) + 3, False)]:
        rng = np.random.default_rng(n)
        cuts = np.sort(rng.integers(0, n + 1, n // 90))
        seg = np.diff(np.concatenate([[0], cuts, [n]]))
        x = rng.integers(-1000, 1000, n).astype(np.int32)
        dx, dseg = gpu_ctx.to_device(x, A.tarray(1, A.i32)), gpu_ctx.to_device(seg, A.tarray(1, Int))
        before = gpu_ctx.flags
        gpu_ctx.flags = before | gpu_ctx.FLAG_DUMP_EXEC
        capfd.readouterr()
        try:
            out = run.execute(dx, dseg)
        finally:
            gpu_ctx.flags = before
        grid = int(re.search(r"acc_foldseg<<<(\d+),256", capfd.readouterr().err).group(1))
        tiles = -(-n // (4096 if half and reads else 8192))
        assert grid == tiles + -(-tiles // 256), n          # and the workgroups that complete ends across tiles
        sums = np.concatenate([[0], np.cumsum(3 * x.astype(np.int64) + 1 if reads else np.full(n, 2, np.int64))])
        ends = np.cumsum(seg)
        want = (sums[ends] - sums[ends - seg]).astype(np.int32)
        assert np.array_equal(out.to_host(), want), n
