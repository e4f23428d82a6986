"""The native calling side (csrc/bz_pycall.cpp) hands the C ABI what ctypes would: every call is bound to a recording function
of the same C signature and made twice, through the native conversion and through the Python one that it falls back to."""
import ctypes as C
import importlib.machinery
import os

import numpy as np
import pytest
import torch

from blitz_scale_amd import _lib
from blitz_scale_amd import kernel as K
from blitz_scale_amd._lib import BZ_LAYOUT_NHD, BzError, BzPagedKV

NAMES = sorted(K._Calls.WHAT)


def _table():
    pt = K.PageTable(3, 16, 8, 128, torch.zeros(64, dtype=torch.bfloat16), layout=BZ_LAYOUT_NHD)
    pt.indices_d = torch.zeros(4, dtype=torch.int32)
    pt.indptr_d, pt.last_page_len_d = pt.indices_d[1:], pt.indices_d[2:]
    return pt


class Bound:
    """The call `name` bound to a function that notes its arguments and returns `status`; `slow` counts the falls back."""

    def __init__(self, name, status=0):
        native, (res, types) = _lib.load_pycall(), _lib.SIGNATURES[name]
        self.types, self.seen, self.slow = types, [], 0

        def record(*args):
            self.seen.append([bytes(C.string_at(a, C.sizeof(BzPagedKV))) if t is _lib._kvp else a for t, a in zip(types, args)])
            return status

        self.fn = C.CFUNCTYPE(res, *types)(record)
        native.setup(torch.Tensor, torch.Tensor.data_ptr, K._DTYPES, K.PageTable, lambda: True, lambda: 5, lambda dev: 0x7000 + dev)
        convert = {"p": K._ptr, "d": K.bz_dtype, "k": lambda t: C.byref(t.as_struct()), "t": int,
                   "s": lambda s: 0x7005 if s is None else int(s)}
        self.spec = native.specs()[name]
        ways = [convert.get(letter, lambda value: value) for letter in self.spec]

        def slowly(*args):
            self.slow += 1
            return self.fn(*[way(a) for way, a in zip(ways, args)])

        self.slowly = slowly
        self.call = native.bind(name, C.cast(self.fn, C.c_void_p).value, slowly, _lib.check, "what")


@pytest.fixture(autouse=True)
def the_real_side_back():
    yield
    K._calls.__dict__.clear()  # the next call binds again, with torch's own functions


def _usual(letter, i):
    return {"p": torch.zeros(8, dtype=torch.float16), "d": torch.zeros(1, dtype=torch.bfloat16), "k": _table(), "u": 7 + i, "i": 2,
            "t": True, "f": 0.1 + i, "s": None}[letter]


@pytest.mark.parametrize("name", NAMES)
def test_usual_arguments_go_through_natively_and_arrive_as_through_ctypes(name):
    b = Bound(name)
    args = [_usual(letter, i) for i, letter in enumerate(b.spec)]
    assert len(args) == len(b.types)
    assert b.call(*args) is None and b.slow == 0
    b.slowly(*args)
    assert b.seen[0] == b.seen[1]


@pytest.mark.parametrize("letter,value,native", [
    ("p", None, True), ("p", 1 << 40, True), ("p", np.int64(4096), False), ("p", torch.nn.Parameter(torch.ones(2)), False),
    ("d", torch.zeros(1, dtype=torch.uint8), True), ("d", torch.zeros(1), True), ("u", -1, True), ("u", np.int32(9), False),
    ("u", 1 << 33, True), ("i", -3, True), ("t", 0, True), ("t", np.bool_(True), False), ("t", 2.0, False), ("f", 3, False),
    ("f", np.float32(0.5), False), ("s", 12345, True), ("s", np.int64(77), False)])
@pytest.mark.parametrize("name", ["bz_decode_step", "bz_store_prefill_kv", "bz_batch_prefill_ragged"])
def test_unusual_arguments_arrive_as_through_ctypes(name, letter, value, native):
    b = Bound(name)
    if letter not in b.spec:
        pytest.skip("no such argument")
    args = [_usual(x, i) for i, x in enumerate(b.spec)]
    args[b.spec.index(letter)] = value
    b.call(*args)
    assert (b.slow == 0) == native
    b.slowly(*args)
    assert b.seen[0] == b.seen[1]


@pytest.mark.parametrize("letter,value,error", [("u", 1.5, C.ArgumentError), ("f", "x", C.ArgumentError), ("d", torch.zeros(1, dtype=torch.int64), KeyError),
                                                ("p", "address", ValueError), ("k", None, AttributeError)])
def test_what_ctypes_refuses_stays_refused(letter, value, error):
    b = Bound("bz_decode_step")
    args = [_usual(x, i) for i, x in enumerate(b.spec)]
    args[b.spec.index(letter)] = value
    with pytest.raises(error):
        b.call(*args)
    with pytest.raises(error):
        b.slowly(*args)
    assert not b.seen


def test_a_table_of_another_kind_and_a_changed_one():
    class Table(K.PageTable):
        def as_struct(self):
            s = super().as_struct()
            s.batch_size = 99
            return s

    b = Bound("bz_append_decode_kv")
    args = [_usual(x, i) for i, x in enumerate(b.spec)]
    b.call(*args)
    args[0].set_layer(3, 100)  # (the struct is made anew for every call)
    args[0].steps_ahead_d = torch.zeros(1, dtype=torch.int32)
    b.call(*args)
    assert b.slow == 0 and b.seen[1][0] == bytes(args[0].as_struct()) != b.seen[0][0]
    own = Table(3, 16, 8, 128, torch.zeros(64, dtype=torch.bfloat16))
    own.indices_d = own.indptr_d = own.last_page_len_d = args[0].indices_d
    b.call(own, *args[1:])
    assert b.slow == 1 and b.seen[2][0] == bytes(own.as_struct())


def test_a_status_is_raised_and_the_number_of_arguments_looked_at():
    b = Bound("bz_rms_norm", status=_lib.BZ_ERR_BAD_ARG)
    args = [_usual(x, i) for i, x in enumerate(b.spec)]
    with pytest.raises(BzError, match="what error"):
        b.call(*args)
    args[3] = torch.nn.Parameter(args[3])
    with pytest.raises(BzError, match="what error"):
        b.call(*args)
    assert b.slow == 1
    with pytest.raises(TypeError):
        b.call(*args[1:])


def test_every_call_is_bound_to_the_library():
    for name in NAMES:
        assert callable(getattr(K._calls, name)) and K._calls.__dict__[name]
    with pytest.raises(BzError):  # (refused on the host, before anything is launched)
        K._calls.bz_silu_and_mul(None, None, torch.zeros(1, dtype=torch.float16), 1, 8, 0)


def test_both_sides_know_the_same_arguments():
    assert _lib.load_pycall().specs() == K._Calls.SPECS


def test_whether_the_gpu_is_up_is_asked_again_after_a_setup():
    b = Bound("bz_rms_norm")
    args = [_usual(x, i) for i, x in enumerate(b.spec)]
    b.call(*args)
    assert b.slow == 0
    _lib.load_pycall().setup(torch.Tensor, torch.Tensor.data_ptr, K._DTYPES, K.PageTable, lambda: False, lambda: 5, lambda dev: 1)
    b.call(*args)
    assert b.slow == 1 and b.seen[0] == b.seen[1]


def test_without_the_native_side_calls_go_through_ctypes(monkeypatch):
    """As on an interpreter that bz_pycall was not built for."""
    suffix = importlib.machinery.EXTENSION_SUFFIXES[0]
    assert _lib.PYCALL_PATH.endswith("bz_pycall" + suffix) and suffix != ".so"
    monkeypatch.setattr(_lib, "PYCALL_PATH", _lib.PYCALL_PATH.replace(suffix, ".cpython-399-other.so"))
    monkeypatch.setattr(_lib, "_pycall", None)
    assert _lib.load_pycall() is None
    K._calls.__dict__.clear()
    x = torch.zeros(8, dtype=torch.float16)
    for name in NAMES:
        assert callable(getattr(K._calls, name))
    with pytest.raises(BzError, match="siluAndMul"):  # (refused on the host, before anything is launched)
        K._calls.bz_silu_and_mul(None, None, x, 1, 8, 0)
    with pytest.raises(TypeError):
        K._calls.bz_silu_and_mul(None, None, x, 1, 8)
    with pytest.raises(C.ArgumentError):
        K._calls.bz_silu_and_mul(x, x, x, 1.5, 8, 0)


def test_building_without_a_compiler_leaves_no_native_side(monkeypatch, tmp_path):
    from blitz_scale_amd import build
    monkeypatch.setattr(build, "LIB_DIR", str(tmp_path))
    assert os.path.basename(build.build_pycall(verbose=False)) == os.path.basename(_lib.PYCALL_PATH)
    monkeypatch.setenv("CXX", str(tmp_path / "no-such-compiler"))
    assert build.build_pycall(verbose=False) is None and not os.listdir(tmp_path)
