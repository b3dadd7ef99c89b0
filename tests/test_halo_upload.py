"""A halo map that is refused leaves the one before it in use."""
import ctypes as C

import numpy as np
import torch

from conftest import mod

native = mod("native")


def _upload(ctx, dst, src):
    ip = C.POINTER(C.c_int32)
    return ctx.lib.nh_upload_halo_map(ctx.handle, dst.ctypes.data_as(ip), src.ctypes.data_as(ip), dst.size)


def test_refused_map_keeps_the_present_one(hostemu_lib):
    case = mod("setup").build_case(glevel=2, vlayer=78, ztop=78000.0, dz_bottom=200.0, dtl=600.0, seed=3)
    ctx = mod("hipdyn").HipContext(case.geo, case.const, device="cpu", lib_path=hostemu_lib)
    ops = mod("ops").HipOperators(ctx)
    f = torch.randn((4, ctx.NF), dtype=torch.float64, generator=torch.Generator().manual_seed(1))

    def outputs():
        filled = f.clone()
        ctx.COMM_data_transfer(filled)
        return filled, ops.divdamp(*f)

    want = outputs()
    # slots x levels past 32 bits, then a column that does not exist
    many = np.full((1 << 31) // case.topo.kall + 1, int(case.topo.halo_dst[0]), dtype=np.int32)
    assert _upload(ctx, many, many) == -1
    bad = np.array([ctx.ncol], dtype=np.int32)
    assert _upload(ctx, bad, bad) == -1
    for a, b in zip(outputs(), want):
        assert torch.equal(a, b)
    # an empty map is none: the calls that need one refuse
    none = np.zeros(0, dtype=np.int32)
    assert _upload(ctx, none, none) == 0
    for call in (lambda: ctx.COMM_data_transfer(f.clone()), lambda: ops.divdamp(*f)):
        try:
            call()
        except RuntimeError as e:
            assert "NH_ERR_STATE" in str(e)
        else:
            raise AssertionError("accepted without a halo map")
    ctx.close()
