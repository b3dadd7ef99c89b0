"""The mixed form's filters against the FP64 form on the same rough fields.

On smooth fields a filter's differences cancel and leave few FP32 digits, so a bound
there says little; on noise of grid scale the n terms of a result are independent and
their absolute values sum to at most sqrt(n) of its 2-norm (Cauchy-Schwarz).  One
pass rounds the input and the coefficient (2 u) and up to 21 partial sums, u = 6e-8:
23 u sqrt(35) = 8e-6 for the damping (7 points of 3 components, 14 of w), less for the
others, and there are two passes: 2e-5."""
import pytest
import torch

from conftest import mod


def _compare(glevel, vlayer, device, lib):
    case = mod("setup").build_case(glevel=glevel, vlayer=vlayer, ztop=1000.0 * vlayer, dz_bottom=200.0, dtl=600.0,
                                   with_state=False)
    out = {}
    for precision in ("float64", "mixed"):
        ctx = mod("hipdyn").HipContext(case.geo, case.const, device=device, lib_path=lib, precision=precision)
        ops = mod("ops").HipOperators(ctx)
        f = torch.randn((16, ctx.NF), generator=torch.Generator().manual_seed(glevel), dtype=torch.float32)
        f[0] = 1.0 + 0.1 * f[0].abs()          # density of prog
        f = f.to(device=ctx.device, dtype=ctx.dtype).contiguous()
        ctx.COMM_data_transfer(f)
        out[precision] = list(ops.hdiffusion(f[:6].contiguous(), f[6:12].contiguous())) + list(ops.divdamp(*f[12:16]))
        ctx.close()
    for n, (a, b) in enumerate(zip(out["float64"], out["mixed"])):
        assert torch.isfinite(b).all() and float(a.norm()) > 0.0
        assert float((a - b.double()).norm() / a.norm()) <= 2e-5, n


@pytest.mark.parametrize("glevel,vlayer", [(3, 9), (4, 12)])
def test_host_mixed_filters(hostemu_lib, glevel, vlayer):
    _compare(glevel, vlayer, "cpu", hostemu_lib)


@pytest.mark.gpu
@pytest.mark.parametrize("glevel,vlayer", [(4, 12), (6, 40), (7, 15)])
def test_gpu_mixed_filters(glevel, vlayer):
    _compare(glevel, vlayer, "cuda:0", None)
