"""Paired passes just below their line (256 clusters in FP64, 512 in
FP32-mixed) against the separate ones, bit for bit, and a run just above it:
the cluster counts say which side a mesh is on (a plan that moved one would
leave nothing compared).
"""
import numpy as np
import pytest

import test_gpu_paired_passes as paired
from weldformfem_amd import WFX_FP32_MIXED, WFX_FP64, workloads

pytestmark = pytest.mark.gpu

LINE = {WFX_FP64: 256, WFX_FP32_MIXED: 512}
# mesh, precision, clusters
CASES = {
    "hexa40x40x40": (lambda: paired.box(40, 40, 40), WFX_FP64, 250),
    "cylinder24": (lambda: workloads.cylinder_tets(cells=24), WFX_FP64, 252),
    "hexa48x51x50": (lambda: paired.box(48, 51, 50), WFX_FP32_MIXED, 480),
    "cylinder30": (lambda: workloads.cylinder_tets(cells=30), WFX_FP32_MIXED, 504),
    "hexa49x49x49, above": (lambda: paired.box(49, 49, 49), WFX_FP32_MIXED, 574),
}


# (FP32-mixed hexahedra above 256 clusters are paired without coupling and with a
# fixed time step only)
@pytest.mark.parametrize("case,option", [(k, o) for k in CASES
                                         for o in ("plain", "jc" if "48" in k else "jc thermal cfl")])
def test_equals_the_separate_passes(monkeypatch, case, option):
    mesh, precision, clusters = CASES[case]
    print(f"case: paired passes at their line, {case}, precision {precision}, {option}", flush=True)
    monkeypatch.setitem(paired.MESHES, case, mesh)
    a, b = paired.make(case, precision, option), paired.make(case, precision, option)
    assert a.get("cluster_count") == clusters
    assert ("above" in case) == (clusters > LINE[precision])
    for n in (7, 4):  # odd and even: both sets of buffers hold the state on the way
        a.runFused(n)
        b.timeFusedPhases(n)
        for f in ("x", "u", "v", "prev_a", "fi", "mdiag", "vol", "p", "tau", "eps", "pl_strain", "T"):
            np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
        if "cfl" in option:
            np.testing.assert_array_equal(a.dtHistory(n), b.dtHistory(n))
