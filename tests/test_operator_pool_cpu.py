"""The buffers of destroyed operators that a context keeps, on the host:
operators destroyed by another thread than the one that makes them."""
from cpu_library import run


def test_destroyed_by_another_thread():
    run("""
import threading
B = Basis.ho(1, 1)
ctx = E.Context(B)
live, mu, bad = set(), threading.Lock(), []
lib, h = E._lib, ctx.h
def work():
    for _ in range(40000):
        op = ctypes.c_void_p()
        assert lib.imsrg_op_create(h, 1, ctypes.byref(op)) == 0
        d = ctypes.cast(op, ctypes.POINTER(ctypes.c_void_p))[1]  # (ctx, buffer, ..)
        with mu:
            if d in live:
                bad.append(d)
            live.add(d)
        with mu:
            live.discard(d)
        assert lib.imsrg_op_destroy(op) == 0
ts = [threading.Thread(target=work) for _ in range(8)]
[t.start() for t in ts]
[t.join() for t in ts]
assert not bad
""", IMSRG_EMU_CHECK=1)
