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


def _outputs(case, state, precision, maps, device, lib):
    """Operators and two steps with each of the halo maps (dst, src, used); used: on a
    context whose workspace another state has been through."""
    out = []
    for dst, src, used in maps:
        ctx = mod("hipdyn").HipContext(case.geo, case.const, device=device, lib_path=lib, precision=precision)
        _upload(ctx, dst, src)
        dyn = mod("hipdyn").HipDynamics(ctx, state)
        ops = mod("ops").HipOperators(ctx)
        if used:
            keep = dyn.prog.clone(), dyn.progq.clone()
            dyn.prog *= 1.5
            ops.hdiffusion(dyn.prog, dyn.prog.clone())
            dyn.dynamics_step()
            dyn.prog, dyn.progq = keep
        res = [ops.divdamp(*dyn.prog[1:5])]
        diag, _ = ops.prepost(dyn.prog.clone(), dyn.progq)
        res.append(ops.hdiffusion(dyn.prog, diag))
        for _ in range(2):
            dyn.dynamics_step()
        res += [dyn.prog.clone(), dyn.progq.clone()]
        ctx.sync()
        ctx.close()
        out.append([r.cpu() for r in res])
    return out


def _same(case, state, precision, maps, device, lib):
    first, *others = _outputs(case, state, precision, maps, device, lib)
    for other in others:
        for x, y in zip(first, other):
            assert torch.isfinite(x).all()
            assert torch.equal(x, y)


def _twice(dst, src):
    return np.append(dst, dst[0]), np.append(src, src[0])


def _partial(precision, device, lib):
    """A map that leaves columns out (no duplicate): read at the source, with the mean
    fluxes copied, one tracer per remap and the cleared hyperdiffusion workspace."""
    case = mod("setup").build_case(glevel=3, vlayer=9, ztop=9000.0, dz_bottom=200.0, dtl=600.0, seed=3)
    state = mod("initial").blob_tracers(case.geo, case.state, ntracer=2, seed=3)
    n = case.topo.halo_dst.size * 2 // 3
    part = np.asarray(case.topo.halo_dst)[:n], np.asarray(case.topo.halo_src)[:n]
    _same(case, state, precision, [(*part, False), (*_twice(*part), False), (*part, True)], device, lib)


def _large(device, lib):
    """8-byte fields of more than 4 million values keep filled halos with a map that
    fills every column: no copy of the mean fluxes, pairs of tracers per remap (whose
    scratch is the hyperdiffusion's), against the map listed with a duplicate."""
    case = mod("setup").build_case(glevel=7, vlayer=22, ztop=22000.0, dz_bottom=200.0, dtl=300.0, seed=3)
    state = mod("initial").blob_tracers(case.geo, case.state, ntracer=2, seed=3)
    full = np.asarray(case.topo.halo_dst), np.asarray(case.topo.halo_src)
    assert state["PROGq"].shape[-1] == 3
    _same(case, state, "float64", [(*full, False), (*_twice(*full), False)], device, lib)


@pytest.mark.parametrize("precision", ["float64", "mixed"])
def test_host_partial_map(hostemu_lib, precision):
    _partial(precision, "cpu", hostemu_lib)


def test_host_large_fields_filled(hostemu_lib):
    _large("cpu", hostemu_lib)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["float64", "mixed"])
def test_gpu_partial_map(precision):
    _partial(precision, "cuda:0", None)


@pytest.mark.gpu
def test_gpu_large_fields_filled():
    _large("cuda:0", None)
