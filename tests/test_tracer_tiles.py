"""Tracer transport against the oracle where the horizontal kernels' tiles, level
chunks and tracer pairs end: narrow regions, level counts off the chunk length,
an odd tracer left over, the limiter on (tiles) and off (points).

One step, FP64.  The mass fluxes agree to about 1e-13 after it (round-off of the
dynamics) and a tracer update is a few dozen operations on them, so 1e-12 of the
largest mass holds."""
import copy

import numpy as np
import pytest

from conftest import mod


def _compare(glevel, vlayer, ntracer, limiter, device, lib):
    from oracle import dynamics as od
    case = mod("setup").build_case(glevel=glevel, vlayer=vlayer, ztop=1000.0 * vlayer, dz_bottom=200.0, dtl=300.0, seed=3)
    const = copy.copy(case.const)
    const.THUBURN_LIM = limiter
    state = mod("initial").blob_tracers(case.geo, case.state, ntracer=ntracer, seed=3)
    ref = od.OracleDynamics(od.OracleContext(case.geo, const, None), state)
    ctx = mod("hipdyn").HipContext(case.geo, const, device=device, lib_path=lib)
    dyn = mod("hipdyn").HipDynamics(ctx, state)
    ref.step()
    dyn.dynamics_step()
    got = dyn.state()
    ctx.close()
    t = case.topo
    s, ks = slice(1, t.gall_1d - 1), slice(1, t.kall - 1)
    for q in range(got["PROGq"].shape[-1]):
        a, b = ref.PROGq[s, s, ks, :, q], got["PROGq"][s, s, ks, :, q]
        ap, bp = ref.PROGq_pl[0, ks, :, q], got["PROGq_pl"][0, ks, :, q]
        scale = max(np.abs(a).max(), np.abs(ap).max())
        assert max(np.abs(a - b).max(), np.abs(ap - bp).max()) <= 1e-12 * scale


@pytest.mark.parametrize("glevel,vlayer,ntracer,limiter", [(2, 5, 1, True), (3, 9, 2, True), (3, 16, 1, False),
                                                           (4, 12, 3, True)])
def test_host_tracer_tiles(hostemu_lib, glevel, vlayer, ntracer, limiter):
    _compare(glevel, vlayer, ntracer, limiter, "cpu", hostemu_lib)


@pytest.mark.gpu
@pytest.mark.parametrize("glevel,vlayer,ntracer,limiter", [(2, 5, 1, True), (4, 29, 2, True), (4, 16, 2, False),
                                                           (6, 6, 1, True)])
def test_gpu_tracer_tiles(glevel, vlayer, ntracer, limiter):
    _compare(glevel, vlayer, ntracer, limiter, "cuda:0", None)
