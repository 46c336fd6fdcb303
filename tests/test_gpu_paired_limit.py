"""Paired passes with two work-groups on a CU (FP32-mixed, 257 to 512 clusters)
against the separate ones, bit for bit, and on both sides of the lines."""
import numpy as np
import pytest

import test_gpu_paired_passes as paired
from weldformfem_amd import WFX_FP32_MIXED, WFX_FP64, workloads

pytestmark = pytest.mark.gpu

MESHES = {
    "hexa40x40x41": lambda: paired.box(40, 40, 41),
    "hexa44x45x46": lambda: paired.box(44, 45, 46),
    "hexa52x50x50": lambda: paired.box(52, 50, 50),
    "cylinder27": lambda: workloads.cylinder_tets(cells=27),
}


@pytest.mark.parametrize("option", ["plain", "jc thermal cfl"])
@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_equals_the_separate_passes(monkeypatch, mesh, precision, option):
    print(f"case: paired passes at their line, {mesh}, precision {precision}, {option}", flush=True)
    monkeypatch.setitem(paired.MESHES, mesh, MESHES[mesh])
    a, b = paired.make(mesh, precision, option), paired.make(mesh, precision, option)
    a.runFused(6)
    b.timeFusedPhases(6)
    for f in ("x", "u", "v", "prev_a", "fi", "mdiag", "vol", "p", "tau", "eps", "pl_strain", "T"):
        np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
