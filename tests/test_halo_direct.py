"""Halo values read at their source against filled halos: the same bits.

A halo map that lists one destination twice (with the same source) describes
the same fill but keeps the library on the filling path, so the two can be
compared on everything that reads halo values inside a step.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from conftest import mod

native = mod("native")


def _upload(ctx, dst, src):
    ip = C.POINTER(C.c_int32)
    dst = np.ascontiguousarray(dst, dtype=np.int32)
    src = np.ascontiguousarray(src, dtype=np.int32)
    native.check(ctx.lib, ctx.lib.nh_upload_halo_map(ctx.handle, dst.ctypes.data_as(ip), src.ctypes.data_as(ip),
                                                     dst.size), "nh_upload_halo_map")


def _run(case, state, precision, fill, device, lib, steps=2):
    ctx = mod("hipdyn").HipContext(case.geo, case.const, device=device, lib_path=lib, precision=precision)
    t = case.topo
    if fill:
        _upload(ctx, np.append(t.halo_dst, t.halo_dst[0]), np.append(t.halo_src, t.halo_src[0]))
    dyn = mod("hipdyn").HipDynamics(ctx, state)
    # a caller's own halo values: the step reads the ones it is given
    dyn.prog[5, :7] *= 1.0 + 1.0e-3
    ops = mod("ops").HipOperators(ctx)
    out = [ops.divdamp(*dyn.prog[1:5])]
    diag, _ = ops.prepost(dyn.prog.clone(), dyn.progq)
    out.append(ops.hdiffusion(dyn.prog, diag))
    for _ in range(steps):
        dyn.dynamics_step()
    out += [dyn.prog.clone(), dyn.progq.clone()]
    ctx.sync()
    ctx.close()
    return [o.cpu() for o in out]


def _compare(precision, vlayer, glevel, device, lib):
    case = mod("setup").build_case(glevel=glevel, vlayer=vlayer, ztop=1000.0 * vlayer, dz_bottom=200.0, dtl=600.0, seed=3)
    state = mod("initial").blob_tracers(case.geo, case.state, ntracer=1, seed=3)
    a = _run(case, state, precision, False, device, lib)
    b = _run(case, state, precision, True, device, lib)
    for x, y in zip(a, b):
        assert torch.isfinite(x).all()
        assert torch.equal(x, y)


@pytest.mark.parametrize("precision", ["float64", "mixed"])
@pytest.mark.parametrize("glevel,vlayer", [(3, 9), (4, 10)])
def test_host_direct_equals_filled(hostemu_lib, precision, glevel, vlayer):
    _compare(precision, vlayer, glevel, "cpu", hostemu_lib)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["float64", "mixed"])
@pytest.mark.parametrize("glevel,vlayer", [(4, 11), (6, 13)])
def test_gpu_direct_equals_filled(precision, glevel, vlayer):
    _compare(precision, vlayer, glevel, "cuda:0", None)
