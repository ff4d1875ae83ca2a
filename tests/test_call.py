"""The native side of the Python calls (csrc/p1a_call.cpp): every argument reaches the C ABI as ctypes would hand it over. The library's
entry points are stood in for by callbacks that note what they get; no GPU."""
import ctypes
import importlib
import os
import subprocess
import sys
import sysconfig
from fractions import Fraction

import numpy as np
import pytest

p1a = importlib.import_module("p100e-engine_amd")
b = importlib.import_module("p100e-engine_amd.binding")
VP, I, F, SZ = ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_size_t
KV = ctypes.POINTER(b.p1a_kv)
SIGNATURES = {"p1a_attn_prep": [VP] * 8 + [KV, I, I, I, I, F, F, I, I, I, VP], "p1a_attn_decode_a16": [VP, KV, VP, VP, VP, I, I, VP, VP, I, I, F, VP],
              "p1a_attn_prefill": [VP, KV, VP, VP, I, I, I, F, VP, SZ, VP], "p1a_kv_append": [KV, VP, VP, I, VP, VP, I, VP]}


class Tensor:
    def __init__(self, at, n=0):
        self.at, self.n = at, n

    def data_ptr(self):
        return self.at

    def numel(self):
        return self.n

    def element_size(self):
        return 4


class Calls(list):
    pass


@pytest.fixture
def calls(monkeypatch):
    got = Calls()

    def stand_in(types):
        def f(*a):
            got.append([{n: getattr(x.contents, n) for n, _ in b.p1a_kv._fields_} if isinstance(x, KV) else x for x in a])
            return 0
        return ctypes.CFUNCTYPE(I, *types)(f)
    kept = got.kept = {n: stand_in(t) for n, t in SIGNATURES.items()}
    m = b._calls()
    m.bind(*(ctypes.cast(kept[n], VP).value for n in SIGNATURES), b.KVCache, lambda: 0x7770, I, ctypes.c_uint32, SZ, F, VP, b.p1a_kv)
    yield got
    b._call = None
    b._calls()                                                 # the library's own entry points again


def test_arguments_reach_the_library(calls):
    big = 0x7fff12345678
    c = p1a.KVCache(p1a.KV_Q8_0, 4096, 4, 256, big, big + 64, Tensor(0x5000), Tensor(0x6000), 8, 1 << 33)
    want = dict(type=8, n_ctx=4096, Hkv=4, D=256, k=big, v=big + 64, pt=0x5000, rtab=0x6000, psh=8, pstride=1 << 33)
    slot = c.slot(3, 17)
    want_slot = dict(want, pt=0x5000 + 4 * 3 * 17, rtab=None)
    flat = p1a.KVCache(p1a.KV_F16, 100, 2, 64, 0x100, 0x200)
    want_flat = dict(type=1, n_ctx=100, Hkv=2, D=64, k=0x100, v=0x200, pt=None, rtab=None, psh=0, pstride=0)
    t = [Tensor(0x1000 + 16 * i) for i in range(8)]
    at = [x.at for x in t]
    p1a.attn_prep(*t, c, -1, 5, 24, 64, 1e6, 1e-6, ldq=7, ldk=8, ldv=9)
    p1a.attn_decode(t[0], slot, t[1], 2, 77, 24, 0.0625)
    p1a.attn_decode_dev(t[0], flat, t[1], 2, t[2], 999, 4, 0.125, gate=t[3])
    p1a.attn_decode_rows(t[0], c, t[1], 4, t[2], 24, 0.5, gate=t[3], rows_per_seq=2, qbuf=t[4])
    p1a.attn_prefill(t[0], slot, t[1], 100, 3, 24, 0.25, gate=t[2], scratch=Tensor(0x9000, 1 << 32))
    p1a.attn_prefill(t[0], flat, t[1], 100, 3, 24, 0.25)
    p1a.kv_append(slot, t[0], t[1], 9, 10)
    p1a.kv_append_dev(c, t[0], t[1], t[2], 10)
    p1a.kv_append_rows(c, t[0], t[1], t[2], 10)
    p1a.attn_decode(t[0], b.KVDesc(slot.struct()), t[1], True, 77, 24, 1)
    f = lambda x: ctypes.c_float(x).value
    s = 0x7770
    assert calls == [
        at + [want, -1, 5, 24, 64, f(1e6), f(1e-6), 7, 8, 9, s],
        [at[0], want_slot, at[1], None, None, 2, 77, None, None, 0, 24, f(0.0625), s],
        [at[0], want_flat, at[1], at[3], None, 2, 0, at[2], None, 0, 4, f(0.125), s],
        [at[0], want, at[1], at[3], at[4], 4, 0, None, at[2], 2, 24, f(0.5), s],
        [at[0], want_slot, at[1], at[2], 100, 3, 24, f(0.25), 0x9000, 1 << 34, s],
        [at[0], want_flat, at[1], None, 100, 3, 24, f(0.25), None, 0, s],
        [want_slot, at[0], at[1], 9, None, None, 10, s],
        [want, at[0], at[1], 0, at[2], None, 10, s],
        [want, at[0], at[1], -1, None, at[2], 10, s],
        [at[0], want_slot, at[1], None, None, 1, 77, None, None, 0, 24, 1.0, s]]


@pytest.mark.parametrize("change", [dict(T=1.5), dict(T=None), dict(q=3), dict(scale="x"), dict(c=object()), dict(c=None)])
def test_what_is_no_argument_is_refused(calls, change):
    a = dict(q=Tensor(16), c=p1a.KVCache(p1a.KV_F16, 100, 2, 64, 0x100, 0x200), out=Tensor(32), T=1, p0=0, Hq=4, scale=1.0)
    with pytest.raises((TypeError, AttributeError, ctypes.ArgumentError)):
        p1a.attn_decode(**{**a, **change})
    assert not calls


class Stands:
    def __init__(self, x):
        self._as_parameter_ = x


class Sub(b.p1a_kv):
    pass


NUMBERS = [3, True, -1, (1 << 40) + 5, np.int32(7), np.int64(-2), np.uint8(200), I(9), I(-9), ctypes.c_long(4), ctypes.c_uint32(4), ctypes.c_short(4), F(2.0), VP(64), Stands(11),
           Stands(Stands(12)), Stands(I(13)), Stands(1.5), 1.5, np.float32(2), np.float64(2), None, "3", b"3", [3], Fraction(3), ctypes.c_size_t(1 << 40)]
REALS = [0.5, 1, True, np.float32(0.25), np.float64(0.75), F(1.5), ctypes.c_double(1.5), I(1), Stands(0.5), Stands(F(2.5)), Fraction(1, 4), None, "0.5", [1.0], 1e300]
ADDRESSES = [0x1000, 0, True, -16, None, VP(0x2000), VP(None), np.int64(0x3000), 1.0, I(5)]


def same(what, by_ctypes, ours, calls):
    """both go through, with the same arguments, or both raise"""
    def go(f):
        del calls[:]
        try:
            f()
        except (TypeError, ctypes.ArgumentError):
            assert not calls
            return "refused"
        return calls[:]
    want = go(by_ctypes)
    assert go(ours) == want, what
    return want != "refused"


def test_arguments_are_taken_as_ctypes_takes_them(calls):
    """ctypes itself is the oracle: the same call through its own prototype and, for the descriptor, its Structure. Whole numbers (cut to
    the parameter's width), ctypes numbers of the very type, what _as_parameter_ stands for; all else refused."""
    ctype = calls.kept
    t = [Tensor(0x1000 + 16 * i) for i in range(8)]
    c = p1a.KVCache(p1a.KV_F16, 100, 2, 64, 0x100, 0x200)
    s, kv = 0x7770, ctypes.byref(c.struct())
    taken = 0
    for x in NUMBERS:                                          # c_int and c_size_t parameters
        taken += same(("T", x), lambda: ctype["p1a_attn_decode_a16"](0x1000, kv, 0x1010, None, None, x, 0, None, None, 0, 4, 1.0, s), lambda: p1a.attn_decode(t[0], c, t[1], x, 0, 4, 1.0), calls)
        same(("bytes", x), lambda: ctype["p1a_attn_prefill"](0x1000, kv, 0x1010, None, 5, 0, 4, 1.0, 0x1020, x, s), lambda: b._calls().prefill(t[0], c, t[1], None, 5, 0, 4, 1.0, t[2], x), calls)
    for x in REALS:
        taken += same(("scale", x), lambda: ctype["p1a_attn_decode_a16"](0x1000, kv, 0x1010, None, None, 1, 0, None, None, 0, 4, x, s), lambda: p1a.attn_decode(t[0], c, t[1], 1, 0, 4, x), calls)
    for x in ADDRESSES:                                        # what data_ptr() gives
        taken += same(("data_ptr", x), lambda: ctype["p1a_attn_decode_a16"](x, kv, 0x1010, None, None, 1, 0, None, None, 0, 4, 1.0, s), lambda: p1a.attn_decode(Tensor(x), c, t[1], 1, 0, 4, 1.0), calls)
    decode = ctype["p1a_attn_decode_a16"]
    fields = [("type", NUMBERS), ("n_ctx", NUMBERS), ("D", NUMBERS), ("psh", NUMBERS), ("pstride", NUMBERS), ("k", ADDRESSES), ("v", ADDRESSES),
              ("pt", [Tensor(x) for x in ADDRESSES] + [None]), ("rtab", [Tensor(x) for x in ADDRESSES] + [None]), ("_pt_off", [0, 5, True, -3, 1 << 33, np.int64(2), I(2), 1.0, None])]
    for name, values in fields:
        for x in values:
            d = p1a.KVCache(p1a.KV_F16, 100, 2, 64, 0x100, 0x200, Tensor(0x5000), None, 4, 4096)
            setattr(d, name, x)
            taken += same((name, x), lambda: decode(0x1000, ctypes.byref(d.struct()), 0x1010, None, None, 1, 0, None, None, 0, 4, 1.0, s), lambda: p1a.attn_decode(t[0], d, t[1], 1, 0, 4, 1.0), calls)
    for x in [c.struct(), Sub(1, 2, 3, 64, 16, 16), bytes(64), bytearray(64), (ctypes.c_uint8 * 64)(), None, 5]:   # what struct() gives
        taken += same(("struct", x), lambda: decode(0x1000, ctypes.byref(x), 0x1010, None, None, 1, 0, None, None, 0, 4, 1.0, s), lambda: p1a.attn_decode(t[0], b.KVDesc(x), t[1], 1, 0, 4, 1.0), calls)
    assert taken > 90


def test_the_binding_alone():
    """binding.py loaded by its path, outside the package, finds its native side as it finds the library, and each of two that are
    loaded keeps its own"""
    code = f"""
import importlib, importlib.util, sys
sys.path.insert(0, {os.path.dirname(os.path.dirname(os.path.abspath(b.__file__)))!r})
spec = importlib.util.spec_from_file_location("alone", {b.__file__!r})
m = importlib.util.module_from_spec(spec)
spec.loader.exec_module(m)
for x in (m, importlib.import_module("p100e-engine_amd.binding")):
    x._stream = lambda: None                                   # (no GPU here)
first = importlib.import_module("p100e-engine_amd.binding")
for x in (first, m, first):                                    # each with its own classes, in turn
    try:
        x.attn_decode(None, x.KVDesc(x.p1a_kv(8, 100, 4, 256, 4096, 4096)), None, 1, 0, 24, 1.0)
    except x.P1AError as e:
        assert "null q/out" in str(e), e
    else:
        assert False
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]


def test_the_native_side_is_named_for_its_python(tmp_path):
    """an extension module without an ABI tag would also be loaded by a Python whose objects are laid out differently"""
    assert b.call_path().endswith(sysconfig.get_config_var("EXT_SUFFIX")) and os.path.exists(b.call_path())
    other = tmp_path / "python"
    other.write_text("#!/bin/sh\ncase \"$2\" in *EXTENSION_SUFFIXES*) echo .cpython-399-other.so ;; *) echo /nowhere ;; esac\n")
    other.chmod(0o755)
    r = subprocess.run(["make", "-n", "-B", "-C", os.path.join(os.path.dirname(b.__file__), "csrc"), f"PYTHON={other}"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "-I/nowhere" in r.stdout and "-o ../_p1a_call.cpython-399-other.so" in r.stdout, r.stdout + r.stderr
