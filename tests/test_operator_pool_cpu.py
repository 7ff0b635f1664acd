"""The buffers of destroyed operators that a context keeps, on the host with a
limit on the device memory in use: an allocation that would have succeeded had
they been freed still does, whichever context asks and whatever for; and
operators destroyed by another thread than the one that makes them."""
import pytest

from cpu_library import run

HOARD = """
lib = E._lib
lib.emu_set_limit.argtypes = [ctypes.c_size_t]
lib.emu_in_use.restype = ctypes.c_size_t
def full():
    lib.emu_set_limit(lib.emu_in_use() + 4096)
B = Basis.ho(2, 1)
ctx = E.Context(B)
other = E.Context(Basis.ho(1, 1))
G, T = ctx.op(-1), ctx.tensor(2, 0)
def hoard():
    ops = [ctx.op(1) for _ in range(60)]
    del ops
"""


@pytest.mark.parametrize("call", ["ctx.tensor(2, 0)", "ctx.bch_tensor(G, T)", "[other.op(1) for _ in range(8)]",
                                  "E.Context(Basis.ho(1, 1))"])
def test_pool_is_given_back(call):
    out = run(HOARD + f"""
hoard()
full()
x = {call}
print("made")
""")
    assert "made" in out


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


def test_tensor_workspace_is_given_back():
    """BCH_TENSOR's work operators, kept for its next call"""
    run(HOARD + """
ctx.bch_tensor(G, T)
full()
U = ctx.tensor(2, 0)
lib.emu_set_limit(2 ** 62)
assert ctx.bch_tensor(G, T) >= 1
""")
