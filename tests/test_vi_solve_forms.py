"""The column solve's forms: the unrolled one (40 levels) keeps its rows in
registers, and each form writes the same bits whichever input it overwrites."""
import os
import re
import subprocess

import pytest
import torch

from conftest import PKG, ROOT, mod

CSRC = os.path.join(ROOT, PKG, "csrc")


@pytest.mark.parametrize("variant", ["nicamhip.hip", "nicamhip_f32.hip"])
def test_unrolled_forms_stay_in_registers(variant, tmp_path):
    """u and gamma of 39 rows take 156 registers of 512: scratch means that the rows'
    loads were all hoisted (FP64 then runs at less than half the speed)."""
    import __graft_entry__ as entry
    if not os.path.exists(entry.HIPCC):
        pytest.skip("no hipcc")
    src = tmp_path / "forms.hip"
    defs = "#define NH_REAL float\n#define NH_VARIANT f32\n" if "f32" in variant else ""
    ns = "f32" if "f32" in variant else "f64"
    src.write_text(f'''{defs}#include "{CSRC}/nh_hipexec.h"
using NHX = nh::HipExec;
#include "{CSRC}/nh_engine.h"
#include "{CSRC}/nh_ops.h"
void forms(nh::HipExec& x, long n) {{
  x.run(nh::{ns}::ViSolveOp<39>{{}}, n);
  x.run(nh::{ns}::ViMainV<39>{{}}, n);
}}
''')
    flags = [f for f in entry.HIP_FLAGS if f != "-shared"]
    r = subprocess.run([entry.HIPCC, *flags, "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-c",
                        "-o", str(tmp_path / "forms.o"), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    seen = set()
    for block in r.stderr.split("Function Name: ")[1:]:
        name = re.search(r"ViSolveOp|ViMainV", block.split()[0])
        if name:
            seen.add(name.group())
            for what in (r"ScratchSize \[bytes/lane\]", "VGPRs Spill"):
                assert int(re.search(what + r": (\d+)", block).group(1)) == 0, (name.group(), what)
    assert seen == {"ViSolveOp", "ViMainV"}


def _overwrite(vlayer, precision, device, lib):
    case = mod("setup").build_case(glevel=2, vlayer=vlayer, ztop=1000.0 * vlayer, dz_bottom=200.0, dtl=600.0,
                                   with_state=False)
    ctx = mod("hipdyn").HipContext(case.geo, case.const, device=device, lib_path=lib, precision=precision)
    ops = mod("ops").HipOperators(ctx)
    gen = torch.Generator().manual_seed(vlayer)
    n = torch.rand((9, ctx.NF), generator=gen, dtype=torch.float64).to(ctx.device)
    scale = [1.0, 1.0, 1.0e5, 1.2, 1.0e-5, 1.0e-3, 1.0]
    f = [(s * (a - 0.5)).to(ctx.dtype) for s, a in zip(scale, n)]
    M = ops.vi_matrix((2.0e5 + 1.0e5 * n[7]).to(ctx.dtype), (n[8] - 0.5).to(ctx.dtype), 200.0)
    want = ops.vi_solve(*f, M, 200.0)
    assert torch.isfinite(want).all()
    for q in range(7):
        g = [a.clone() for a in f]
        assert torch.equal(ops.vi_solve(*g, M, 200.0, out=g[q]), want), q
    ctx.close()


# 39 unknowns run unrolled; 2, 4, 5 and 77 rolled by four (the fewest, exact, one over, the most)
SHAPES = [(3, "float64"), (5, "float64"), (6, "mixed"), (40, "float64"), (40, "mixed"), (78, "float64")]


@pytest.mark.parametrize("vlayer,precision", SHAPES)
def test_host_output_over_any_input(hostemu_lib, vlayer, precision):
    _overwrite(vlayer, precision, "cpu", hostemu_lib)


@pytest.mark.gpu
@pytest.mark.parametrize("vlayer,precision", SHAPES)
def test_gpu_output_over_any_input(vlayer, precision):
    _overwrite(vlayer, precision, "cuda:0", None)
