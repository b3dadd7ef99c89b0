"""The tracers of a step do not depend on each other: a step with many (vertical
half steps in groups, one thread per column and tracer) gives each the bits it
has alone beside qv."""
import pytest
import torch

from conftest import mod


def _step(case, state, precision, device, lib, progq=None):
    ctx = mod("hipdyn").HipContext(case.geo, case.const, device=device, lib_path=lib, precision=precision)
    dyn = mod("hipdyn").HipDynamics(ctx, state)
    if progq is not None:
        dyn.progq = progq.to(dyn.prog.device).contiguous()
    q0 = dyn.progq.clone()
    dyn.dynamics_step()
    ctx.sync()
    out = dyn.progq.cpu()
    ctx.close()
    return q0.cpu(), out


def _check(precision, vlayer, ntracer, device, lib):
    case = mod("setup").build_case(glevel=3, vlayer=vlayer, ztop=1000.0 * vlayer, dz_bottom=200.0, dtl=600.0, seed=2)
    state = mod("initial").blob_tracers(case.geo, case.state, ntracer=ntracer, seed=2)
    q0, many = _step(case, state, precision, device, lib)
    assert torch.isfinite(many).all() and not torch.equal(q0[1], many[1])
    for n in (1, ntracer // 2, ntracer):
        _, alone = _step(case, state, precision, device, lib, q0[[0, n]])
        assert torch.equal(alone[1], many[n])


# group of six: below, whole, one over, two groups and a remainder
@pytest.mark.parametrize("precision,vlayer,ntracer", [("float64", 9, 4), ("mixed", 9, 5), ("float64", 12, 6),
                                                      ("mixed", 8, 13)])
def test_host_tracer_groups(hostemu_lib, precision, vlayer, ntracer):
    _check(precision, vlayer, ntracer, "cpu", hostemu_lib)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,vlayer,ntracer", [("float64", 9, 6), ("mixed", 41, 13)])
def test_gpu_tracer_groups(precision, vlayer, ntracer):
    _check(precision, vlayer, ntracer, "cuda:0", None)
