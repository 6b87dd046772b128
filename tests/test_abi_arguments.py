"""Every exported function that takes arguments has them declared to ctypes: undeclared, a pointer passed as a Python integer is
cut to 32 bits."""
from slowrun_amd import _lib


def test_argument_types_are_declared():
    lib = _lib.lib()
    undeclared = [n for n in _lib.EXPORTS if getattr(lib, n).argtypes is None]
    assert set(undeclared) <= {"sce_version", "sce_last_error"}, undeclared
