"""The native caller against ctypes: every order of integers and fp32 numbers, errors, arguments and functions it hands back to ctypes."""
import ctypes as C
import random

import pytest

from nanovllm import _hip

hostpath = pytest.importorskip("nanovllm._hostpath")
i32, i64, u64, f32, vp = _hip.i32, _hip.i64, _hip.u64, _hip.f32, _hip.vp


class Handle:
    pass


def library(signatures, results):
    """Functions that note their arguments; `results`: name -> what it returns."""
    handle, seen = Handle(), []
    for name, (res, args) in signatures.items():
        def note(*got, name=name):
            seen.append((name, got))
            return results.get(name, 0)
        setattr(handle, name, C.CFUNCTYPE(res, *args)(note))
    return handle, seen


def test_every_order_of_kinds():
    rng = random.Random(0)
    signatures = {}
    for n in list(range(0, 16)) + [30, 46, 54] * 8:
        kinds = [f32] * min(n // 3, 8)
        kinds += [rng.choice((vp, i64, i32, u64)) for _ in range(min(n - len(kinds), 46))]
        rng.shuffle(kinds)
        signatures[f"f{len(signatures)}"] = (i32, kinds)
    handle, seen = library(signatures, {})
    call = _hip.native_caller(handle, signatures, _hip.check)
    for name, (_, kinds) in signatures.items():
        args = [rng.choice((0.0, -1.5, 3, 2.0 ** 40)) if k is f32 else {i32: rng.randint(-2 ** 31, 2 ** 31 - 1), i64: rng.randint(-2 ** 63, 2 ** 63 - 1),
                u64: rng.randint(0, 2 ** 64 - 1), vp: rng.choice((None, 0, 0x7fff12345678))}[k] for k in kinds]
        assert call(name, *args) is None
        got = seen.pop()
        assert got[0] == name and [g or 0 for g in got[1]] == [(float(a) if k is f32 else a) or 0 for a, k in zip(args, kinds)]


def test_errors_and_fallback():
    class Error(Exception):
        pass

    def check(code, name):
        if code:
            raise Error(code, name)
    signatures = {"fails": (i32, [i64]), "wide": (i64, [i64]), "text": (i32, [C.c_char_p, i64]), "many": (i32, [i64] * 60), "plain": (i32, [vp, f32])}
    handle, seen = library(signatures, {"fails": -3, "text": 5})
    call = _hip.native_caller(handle, signatures, check)
    with pytest.raises(Error) as e:
        call("fails", 1)
    assert e.value.args == (-3, "fails")
    with pytest.raises(Error):
        call("text", b"abc", 1)                              # (a type that the native path does not take)
    assert seen[-1] == ("text", (b"abc", 1))
    call("many", *range(60))
    assert seen[-1] == ("many", tuple(range(60)))
    call("plain", C.c_void_p(16), 2.0)                       # (an argument that only ctypes converts)
    assert seen[-1] == ("plain", (16, 2.0))
    for bad in ((1,), (1, "x"), (1.5, 2.0)):
        with pytest.raises((TypeError, C.ArgumentError)):
            call("plain", *bad)
    with pytest.raises(AttributeError):
        call("nobody", 1)
    with pytest.raises(TypeError):
        call()


def test_what_ctypes_refuses_stays_refused():
    """None is a null pointer and no integer, and a number has to fit a double: the function is not called."""
    signatures = {"f": (i32, [vp, i64, i32, u64, f32])}
    handle, seen = library(signatures, {})
    call = _hip.native_caller(handle, signatures, _hip.check)
    good = (None, 1, 2, 3, 4.0)
    call("f", *good)
    assert seen.pop() == ("f", good)
    for at, bad in ((1, None), (2, None), (3, None), (4, None), (4, 10 ** 400)):
        args = good[:at] + (bad,) + good[at + 1:]
        with pytest.raises(C.ArgumentError):
            handle.f(*args)
        with pytest.raises(C.ArgumentError):
            call("f", *args)
    assert not seen
