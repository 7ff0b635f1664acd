"""The FP64 tile shapes go by the basis alone.  On the host a launch's time is its
number of workgroups, so a choice by the clock takes the larger tiles, whose sums
round differently from the other shape's and from the merged forms'."""
from cpu_library import run


def test_bits_do_not_depend_on_a_clock():
    run("""
B = Basis.ho(3, 1)
L, R = random_operator(B, -1, 1), random_operator(B, 1, 2)
def commutator(pin):
    ctx = E.Context(B)
    if pin:
        ctx.set_tile_shapes(0, 0)
    return ctx.commutator(ctx.op(-1, L), ctx.op(1, R), mask=E.TALL & ~E.T122).download()
assert np.array_equal(commutator(False), commutator(True))
""")


def test_shapes_reported():
    """unset before the first commutator, then the rule's, in the fused form as in the separate one"""
    run("""
for mask in (E.TALL, E.TALL & ~E.T122):
    B = Basis.ho(1, 1)
    ctx = E.Context(B)
    L, R = ctx.op(-1, random_operator(B, -1, 1)), ctx.op(1, random_operator(B, 1, 2))
    assert (ctx.tuning()["pphh"], ctx.tuning()["ph"]) == ("untuned", "untuned")
    ctx.commutator(L, R, mask=mask)
    assert (ctx.tuning()["pphh"], ctx.tuning()["ph"]) == ("64x64", "64x64")
    ctx.set_tile_shapes(1, 1)
    ctx.commutator(L, R, mask=mask)
    assert (ctx.tuning()["pphh"], ctx.tuning()["ph"]) == ("128x64", "128x64")
""")
