"""The call module next to the ctypes binding: the same argument forms are
taken and refused through either, and the package works without the module.
(Host side only: zero rows, nothing is launched.)"""
import ctypes
import pathlib
import sysconfig

import numpy as np
import pytest

from t2h import _build, _lib

BASE = [None, None, 0, 1536, 0, 1e-6, 0, None, None, 1536, None, 1, 0, None]


class Index:
    def __index__(self):
        return 0


FORMS = [np.int64(0), 0.0, None, "x", b"x", Index(), np.float32(1e-6), 1 << 70, -1, True, ctypes.c_int64(0),
         ctypes.c_int32(0), ctypes.c_void_p(0), (ctypes.c_float * 2)(), ctypes.c_float(1.0),
         ctypes.byref(ctypes.c_int(0)), 10 ** 400, np.zeros(2, np.int64)]


def _outcome(f, args):
    try:
        return f(*args)
    except Exception as e:      # noqa: BLE001 (the kind of error is what is compared)
        return type(e)


@pytest.mark.parametrize("slot", [0, 2, 4, 5], ids=["pointer", "int64", "int32", "float"])
@pytest.mark.parametrize("form", FORMS, ids=lambda v: type(v).__name__)
def test_argument_forms_as_ctypes(slot, form):
    L = _lib.load()
    args = list(BASE)
    args[slot] = form
    want = _outcome(L.t2h_ln_modulate, args)
    if isinstance(want, int):
        want = _outcome(_lib.check, (want,))
    assert _outcome(_lib.call, ("t2h_ln_modulate", *args)) == want


def test_argument_count_as_ctypes():
    L = _lib.load()
    for args in (BASE[:-1], [*BASE, 0]):
        want = _outcome(L.t2h_ln_modulate, args)
        assert _outcome(_lib.call, ("t2h_ln_modulate", *args)) == (None if want == 0 else want)


def test_the_module_is_this_interpreters():
    assert _build.PYCALL_PATH.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    assert ".so" != sysconfig.get_config_var("EXT_SUFFIX")


def test_loads_without_the_module_and_from_a_path_object(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_calls", {})
    monkeypatch.setattr(_lib, "PYCALL_PATH", _build.PYCALL_PATH + ".missing")
    L = _lib.load(pathlib.Path(_build.LIB_PATH))
    assert _lib._calls["t2h_ln_modulate"] is L.t2h_ln_modulate
    _lib.call("t2h_ln_modulate", *BASE)
    bad = list(BASE)
    bad[3] = -1
    with pytest.raises(ValueError, match="bad shape"):
        _lib.call("t2h_ln_modulate", *bad)
