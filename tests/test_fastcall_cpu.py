"""capi's calls through _fastcall against the same calls through ctypes.

Only calls that launch nothing (empty problems and refused arguments), so no
GPU is needed.
"""
import ctypes
import os
import subprocess
import sys
import sysconfig

import numpy as np
import pytest

import fast_dl_amd.capi as capi
# (built with the library: one that is missing or does not load is a failure)
from fast_dl_amd import _fastcall as fastcall

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

EMPTY_GEMM = (0, 0, 0, 4, 4, None, 4, 0, None, 4, 0, None, 4, 0, 1, None, None, 0)
# calls of every argument kind: ints, pointers as int and None, floats, sizes
CALLS = [
    ("sgemm_ex", EMPTY_GEMM + (0,)),
    ("sgemm_ex_select", EMPTY_GEMM + (-1, 0)),
    ("sgemm_ex_ws", EMPTY_GEMM + ((1 << 63) + 16, (1 << 64) - 16, None)),
    ("sgemm_ex_noalloc", EMPTY_GEMM + (None,)),
    ("gemm", (None, None, None, 2, -1, 2)),
    ("gemm", (16, 16, 16, 0, 1, 2)),
    ("add_row_bias", (None, None, 0, 7, 0)),
    ("relu", (None, None, 5, None)),
    ("relu", (None, None, -1, 0)),
    ("relu_backward", (0, 0, 0, 0, 0)),
    ("colsum", (None, None, 3, 3, None)),
    ("softmax", (16, 16, 0, 3, 0)),
    ("softmax_xent", (16, 16, 16, 16, 4, 0, None)),
    ("sgd_update", (None, None, 0.5, 0, 0)),
    ("sgd_update", (None, None, 1, 3, 0)),           # an int where C has a float
    ("idx_gather", (None, None, 4, 4, None, 0, 255.0, None, None, None)),
    ("idx_gather", (16, 16, 4, 4, None, 2, float("inf"), 16, 16, None)),
    ("mlp2_train_step", (None, None, 0, 1, 1, 1, None, None, None, None, 0.1) + (None,) * 11),
    ("relu", (None, None, (1 << 63) + 5, 0)),        # past int64: as ctypes takes it
    ("relu", (ctypes.c_void_p(16), None, 0, 0)),     # a ctypes pointer
    ("relu", (None, None, np.int64(0), 0)),
    ("relu", (None, None, True, 0)),
    ("relu", (None, None, 1.5, 0)),
    ("relu", (None, None)),
    ("relu", (-1, None, 0, 0)),
]


def _outcome(call):
    try:
        return call()
    except Exception as e:  # noqa: BLE001 -- the kind and text are what is compared
        return type(e), str(e)


@pytest.mark.parametrize("name,args", CALLS)
def test_as_ctypes(name, args):
    lib = capi.load_library()

    def through_ctypes():
        status = getattr(lib, "fdl_" + name)(*args)
        if status != 0:
            raise capi.FdlError("fdl_" + name, status, capi.last_error())
        return status

    call = getattr(capi, name)
    assert type(call).__name__ == "builtin_function_or_method"
    assert _outcome(lambda: call(*args)) == _outcome(through_ctypes)


def test_library_loads_on_the_first_call():
    # importing capi loads nothing; the first call loads the library and works
    code = ("import fast_dl_amd.capi as c\n"
            "assert c._LIB is None\n"
            "assert c.relu(None, None, 0, 0) == 0 and c._LIB is not None\n"
            "assert c.relu(None, None, 0, 0) == 0\n")
    subprocess.run([sys.executable, "-c", code], cwd=ROOT, check=True, timeout=120)


def test_module_carries_this_pythons_abi_tag():
    assert os.path.basename(fastcall.__file__) == \
        "_fastcall" + sysconfig.get_config_var("EXT_SUFFIX")
