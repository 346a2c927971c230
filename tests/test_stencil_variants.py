"""Which stencils the code generator gives a variant of their own, compile-only (gfx950, no GPU)."""
import os
import re

import pytest

from accelerate_amd import hip, ir as A


def test_functions_undefined_for_some_values_stay_with_lds(cc_ctx):
    """Lanes in the margins compute on values that are no taps of any element: a function that divides by a tap
    must not."""
    def prog(fn):
        row = A.sunit(3, A.i32)
        sr = A.stup(*[A.stup(row, row, row)] * 3)

        def f(st):
            taps = [t for p in A.untup(st) for r in A.untup(p) for t in A.untup(r)]
            acc = taps[0]
            for t in taps[1:]:
                acc = fn(acc, t)
            return acc

        return A.alam([A.tarray(3, A.i32)], lambda g: A.stencil(sr, A.i32, A.lam([A.stencil_type(sr)], f), A.clamp, g))

    third = lambda a: A.quot(A.i32, a, A.const(A.i32, 3))
    for fn, rows in [(lambda a, t: A.add(A.i32, a, t), True), (lambda a, t: A.add(A.i32, third(a), t), True),
                     (lambda a, t: A.quot(A.i32, a, t), False), (lambda a, t: A.add(A.i32, A.mod(A.i32, a, A.const(A.i32, 0)), t), False)]:
        keys = {}
        for on in (0, 2):
            old = cc_ctx.set_knob("stencil_rows3d", on)
            try:
                keys[on] = cc_ctx.compile(prog(fn)).kernel_keys
            finally:
                cc_ctx.set_knob("stencil_rows3d", old)
        assert (keys[0] != keys[2]) == rows


def _sum(ts):
    acc = ts[0]
    for t in ts[1:]:
        acc = A.add(A.f32, acc, t)
    return acc


_some = lambda t: [t[k] for k in (4, 10, 12, 13, 14, 16, 22)]
_sin = lambda e: A.sin(A.f32, e)
STAGED = {
    # plane after plane, handing on at most three values
    "sum": (lambda t: _sum(t), "planes"),
    "sum_of_sums": (lambda t: _sum([_sum(t[:9]), _sum(t[9:18]), _sum(t[18:])]), "planes"),
    "one_tap": (lambda t: t[13], "planes"),
    "no_tap": (lambda t: A.const(A.f32, 3), "planes"),
    "three_from_the_last_plane_on": (lambda t: _sum([t[26], t[13], t[0]]), "planes"),
    "bound": (lambda t: A.let(A.f32, _sum(t[:2]), lambda x: A.mul(A.f32, x, A.add(A.f32, x, t[26]))), "planes"),
    # back to front: all taps of the earlier planes would have to be handed on
    "backward": (lambda t: _sum(t[::-1]), "rows"),
    "four_products_across": (lambda t: _sum([A.mul(A.f32, t[k], t[k + 18]) for k in range(4)]), "rows"),
    "comparison": (lambda t: A.cond(A.lt(A.f32, t[0], t[13]), t[13], t[26]), "rows"),
    # heavy functions: the kernel would hold them a hundred times
    "sine_of_the_sum": (lambda t: _sin(_sum(t)), "planes"),
    "square_roots": (lambda t: _sum([A.sqrt(A.f32, x) for x in t]), "planes"),
    "two_sines": (lambda t: _sum([_sin(t[4]), t[13], _sin(t[22])]), "rows"),
    "sines": (lambda t: _sum([_sin(x) for x in _some(t)]), "rows"),
}


@pytest.mark.parametrize("name", sorted(STAGED))
def test_functions_taken_plane_by_plane(capfd, name):
    """with register kernels for any number of taps; the generated source says which it is"""
    fn, kind = STAGED[name]
    row = A.sunit(3, A.f32)
    sr = A.stup(*[A.stup(row, row, row)] * 3)
    f = lambda st: fn([t for p in A.untup(st) for r in A.untup(p) for t in A.untup(r)])
    ctx = hip.Context(-1)
    try:
        ctx.set_knob("stencil_rows3d", 2)
        ctx.flags = ctx.flags | ctx.FLAG_DUMP_CC
        capfd.readouterr()
        ctx.compile(A.alam([A.tarray(3, A.f32)], lambda g: A.stencil(sr, A.f32, A.lam([A.stencil_type(sr)], f), A.clamp, g)))
        source = capfd.readouterr().err
    finally:
        ctx.close()
    assert [k for k in ("planes", "rows") if "acc_stencil3d_%s(" % k in source] == [kind]


def test_moves_between_lanes_are_folded_in_one_place():
    """A wave shift without an old value may become a modifier of the operation that uses it, which is known to be right behind
    floating-point operations only: acc_neighbour is the one place that makes such a shift, and asks for the type."""
    device = os.path.join(os.path.dirname(hip.LIB_PATH), "csrc", "device")
    made = {}
    for name in os.listdir(device):
        with open(os.path.join(device, name)) as f:
            text = f.read()
        n = len(re.findall(r"__builtin_amdgcn_(?:update|mov)_dpp\w*\((?!\(int\)(\w+\[k\]), \(int\)\1)", text))
        if n:
            made[name] = n
    assert made == {"prelude.hpp": 1}
