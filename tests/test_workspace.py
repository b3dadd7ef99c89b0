"""Device memory a context takes for its step workspace: 91 fields in the field
precision and 5 in FP64.  Each field more refuses the largest grids that fit today."""
import ctypes as C

import pytest

from conftest import mod

native = mod("native")


@pytest.mark.parametrize("precision,size", [(native.PREC_FP64, 8), (native.PREC_MIXED, 4)])
def test_workspace_fields(hostemu_lib, precision, size):
    lib = native.load(hostemu_lib)
    # far past any address space, so that the refusal states the size
    dims = native.NhDims((1 << 20) + 2, 80, 1, 78, 10)
    consts = native.NhConsts(*([1.0] * 11))
    h = C.c_void_p()
    assert lib.nh_create_ex(C.byref(dims), C.byref(consts), 0, precision, C.byref(h)) == -3
    text = lib.nh_last_error().decode()
    nbytes = int(text.split("workspace allocation of ")[1].split()[0])
    assert nbytes == (91 * size + 5 * 8) * int(lib.nh_field_size(C.byref(dims)))


@pytest.mark.gpu
def test_refused_context_leaves_no_error_behind():
    import torch
    lib = native.load()
    dims = native.NhDims((1 << 20) + 2, 80, 1, 78, 10)
    consts = native.NhConsts(*([1.0] * 11))
    h = C.c_void_p()
    x = torch.ones(1000, device="cuda:0")
    assert lib.nh_create_ex(C.byref(dims), C.byref(consts), 0, native.PREC_FP64, C.byref(h)) == -3
    # torch checks the runtime's pending error after each of its launches
    assert float((x * 2.0).sum()) == 2000.0
