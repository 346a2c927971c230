"""Which stencils the code generator gives a variant of their own, compile-only (gfx950, no GPU)."""
from accelerate_amd import ir as A


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
