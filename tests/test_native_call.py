"""Launchers called without ctypes (``csrc/host/ome_call.cpp``): the arguments that arrive, what goes to ctypes, and errors."""
import ctypes as C

import pytest

from ome_amd.ops import _native as N

pytestmark = pytest.mark.skipif(N._caller is None, reason="built without Python.h")
TYPES = {"p": C.c_void_p, "i": C.c_int, "l": C.c_int64, "f": C.c_float}


def _bind(name, kinds, rc=0):
    got = []
    f = C.CFUNCTYPE(C.c_int, *[TYPES[k] for k in kinds])(lambda *a: (got.append(a), rc)[1])
    assert N._caller.bind(name, C.cast(f, C.c_void_p).value, kinds)
    return f, got


@pytest.mark.parametrize("kinds", ["", "i", "ppllii", "f", "pfi" * 5, "ffffffff" + "i" * 7, "l" * 24, "l" * 25, "plif" * 8, "ipl" * 14 + "ff", "l" * 64 + "f" * 8],
                         ids=lambda k: "%dx%d" % (len(k), k.count("f")))
def test_arguments_arrive(kinds):
    """Six integers in registers, the others on the stack (up to 18, up to 58), eight floats beside them."""
    f, got = _bind("t", kinds)
    edge = {"p": [None, 1, (1 << 47) + 16, 1 << 63], "i": [0, -1, 2**31 - 1, -2**31], "l": [0, -1, 2**63 - 1, -2**63], "f": [0.0, -1.5, 1e-30, 3.0e38]}
    args = [edge[k][i % 4] for i, k in enumerate(kinds)]
    N._caller.call("t", *args)
    want = [C.c_float(a).value if k == "f" else a for a, k in zip(args, kinds)]
    assert got == [tuple(want)]


@pytest.mark.parametrize("args", [(1,), (1, 2, 3), (1.0, 2), (None, 2), ("x", 2), (C.c_int(1), 2)], ids=str)
def test_other_arguments_go_to_ctypes(monkeypatch, args):
    f, got = _bind("t", "ii")
    seen = []
    N._caller.hooks(lambda *a: seen.append(a), N._fail)
    try:
        N._caller.call("t", *args)
        N._caller.call("nothing of that name")
    finally:
        N._caller.hooks(N._slow_call, N._fail)
    assert got == [] and seen == [("t", *args), ("nothing of that name",)]


def test_a_launcher_of_another_library():
    """``lib`` names it, as it does where ctypes makes every call."""
    with pytest.raises(N.NativeError, match="nowhere"):
        N.call("t", 1, lib="nowhere")
    f, got = _bind("ome_ep_handle", "i")
    seen = []
    N._caller.hooks(lambda *a, **kw: seen.append((a, kw)), N._fail)
    try:
        N.call("ome_ep_handle", 1, lib="ome_comm")
    finally:
        N._caller.hooks(N._slow_call, N._fail)
    assert got == [] and seen == [(("ome_ep_handle", 1), {"lib": "ome_comm"})]


def test_a_code_raises():
    f, got = _bind("t", "l", rc=-3)
    with pytest.raises(N.NativeError, match="t failed with code -3"):
        N._caller.call("t", 5)
    assert got == [(5,)]


def test_too_many_for_the_prototype_stay_with_ctypes():
    assert not N._caller.bind("t", 1, "f" * 9) and not N._caller.bind("t", 1, "l" * 65)


def test_every_launcher_can_be_bound():
    for argt in N._SIGNATURES["ome_kernels"].values():
        kinds = [N._KINDS[a] for a in argt]
        assert kinds.count("f") <= 8 and len(kinds) - kinds.count("f") <= 64
