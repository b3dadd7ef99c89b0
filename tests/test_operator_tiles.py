"""Gradient, divergence and Laplacian tiles against the oracle, bit for bit in FP64
(the same products summed in the same order), at tile shapes and level counts
on both sides of the tile width (64 points) and of the levels per chunk."""
import numpy as np
import pytest
import torch

from conftest import mod


def _compare(glevel, vlayer, device, lib):
    from oracle import dynamics as od
    case = mod("setup").build_case(glevel=glevel, vlayer=vlayer, ztop=1000.0 * vlayer, dz_bottom=200.0, dtl=600.0, seed=3)
    layout = mod("layout")
    ctx = mod("hipdyn").HipContext(case.geo, case.const, device=device, lib_path=lib)
    t = case.topo
    g, kall, L = t.gall_1d, t.kall, t.lall
    octx = od.OracleContext(case.geo, case.const, None)
    rng = np.random.default_rng(glevel * 100 + vlayer)
    F = [(rng.standard_normal((g, g, kall, L)), rng.standard_normal((6, kall, 2))) for _ in range(3)]
    T = [torch.from_numpy(layout.pack1(a, b)).to(device) for a, b in F]
    lap, grad = od.laplacian(octx, *F[0]), od.gradient(octx, *F[0])
    div = od.divergence(octx, F[0][0], F[1][0], F[2][0], F[0][1], F[1][1], F[2][1])
    G = ctx.OPRT_gradient(T[0])
    got = [ctx.OPRT_laplacian(T[0]), G[0], G[1], G[2], ctx.divergence(*T)]
    want = [lap] + [(grad[0][..., q], grad[1][..., q]) for q in range(3)] + [div]
    s = slice(1, g - 1)
    for a, (reg, pole) in zip(got, want):
        x, xp = layout.unpack1(a.cpu().numpy(), g, kall, L)
        assert np.array_equal(x[s, s], reg[s, s]) and np.array_equal(xp[0], pole[0])
    ctx.close()


@pytest.mark.parametrize("glevel,vlayer", [(2, 5), (3, 9), (4, 29)])
def test_host_operator_tiles(hostemu_lib, glevel, vlayer):
    _compare(glevel, vlayer, "cpu", hostemu_lib)


@pytest.mark.gpu
@pytest.mark.parametrize("glevel,vlayer", [(2, 5), (4, 29), (6, 13), (7, 6)])
def test_gpu_operator_tiles(glevel, vlayer):
    _compare(glevel, vlayer, "cuda:0", None)
