"""smat_amd.spmm from the extension module against the same function in Python: what they refuse, and with what, for calls that never reach a device."""
import inspect

import pytest

import smat_amd
from smat_amd import host

_call = pytest.importorskip("smat_amd._call")


class Array:
    def __init__(self, address=4096):
        self.address = address

    def data_ptr(self):
        return self.address


class Plain(int):
    pass


A = Array()
OK = (A, A, A, A, A, 16, 8, 16, 1)


def outcome(f, args, kwargs):
    try:
        return f(*args, **kwargs)
    except Exception as e:
        return type(e), str(e).replace("spmm()", "")


def in_python():
    """The function that host.py defines, which the module calls for what it does not take itself."""
    ns = {k: v for k, v in vars(host).items() if not k.startswith("__")}
    src = inspect.getsource(host)
    start = src.index("def spmm(")
    exec(src[start:src.index("\ntry:\n    from . import _call")], ns)
    return ns["spmm"]


@pytest.mark.parametrize("args,kwargs", [
    ((A, A, A, A, A, 16, 7, 16, 1), {}),                                   # the library refuses: N
    ((A, A, A, A, A, 15, 8, 16, 1), {"drop_in": True}),
    ((A, A, A, Array(4097), A, 16, 8, 16, 1), {"c_f32": True}),           # alignment
    ((A, None, A, A, A, 16, 8, 16, 1), {}),                                # NULL
    ((None, A, None, A, A, 16, 8, 16, 3), {"stream": 7}),
    ((A, A, A, A, Array(0), 16, 8, 16, 1), {"stream": None}),
    (OK, {"kernel": 99}),
    (OK, {"kernel": smat_amd.KERNEL_COMPACT}),
    (OK, {"kernel": smat_amd.KERNEL_ROWWISE, "b_row_major": True}),
    (OK, {"plan": None, "kernel": smat_amd.KERNEL_MIXED, "c_f32": 1}),    # flags that are no truth values
    ((A, A, A, A, A, 16, 8, 16), {"nnzb": Plain(1), "kernel": 99}),
    ((A, A, A, A, A, -16, 8, 16, 1), {"kernel": 99}),
    ((A, A, A, A, A, 16, 8.0, 16, 1), {}),                                 # ctypes refuses
    (OK, {"kernel": 2 ** 40}),
    ((A, A, A, 3, A, 16, 8, 16, 1), {}),                                   # no data_ptr
    ((A, A, A, Array("x"), A, 16, 8, 16, 1), {}),
    ((A, A), {}),                                                          # Python refuses
    (OK + (None,) * 7, {}),
    (OK, {"colour": 1}),
    (OK, {"vals": A}),
    (OK, {"plan": 5}),
])
def test_refused_as_in_python(args, kwargs):
    want = outcome(in_python(), args, kwargs)
    assert isinstance(want, tuple)
    assert outcome(smat_amd.spmm, args, kwargs) == want


def test_signature():
    assert smat_amd.spmm is _call.spmm
    assert inspect.signature(smat_amd.spmm) == inspect.signature(in_python())
