"""Clusters with equal tables share them: a structured block, whose clusters
share a handful, against the same block with its nodes renumbered at random,
whose clusters share none.  Neither the element order nor any order of
summation depends on the node numbers, so the results are the same bit for
bit; both kinds of passes, both precisions, block sizes split evenly and cut
into runs, tetrahedra, and two blocks."""
import numpy as np
import pytest

from weldformfem_amd import WFX_FP32_MIXED, WFX_FP64, Domain, workloads

pytestmark = pytest.mark.gpu


def two_blocks():
    x, el = workloads.hexa_box(21, 17, 13, 0.05)
    y, fl = workloads.hexa_box(21, 17, 13, 0.05, (3.0, 0.0, 0.0))
    return np.r_[x, y], np.r_[el, fl + len(x)].astype(np.int32)


MESHES = {
    "evenly split": lambda: workloads.hexa_box(26, 22, 18, 0.05),
    "runs": lambda: workloads.hexa_box(37, 11, 7, 0.05),
    "column": lambda: workloads.hexa_box(1, 1, 700, 0.05),
    "two blocks": two_blocks,
    "tetrahedra": lambda: workloads.cylinder_tets(cells=6)[:2],
}


def make(x, el, bottom, top, v, precision):
    d = Domain(precision)
    d.CreateFromMesh(x, el, el.shape[1])
    d.setDensity(7850.0)
    d.setMaterial(0, 200e9, 0.3, 7850.0, 50e6, 1e9, 0.0)
    for nd in bottom:
        d.AddBCVelNode(int(nd), 2, 0.0)
    for nd in top:
        d.AddBCVelNode(int(nd), 2, -8.0)
    d.AllocateBCs()
    d.set("hg_coeff", 0.06)
    d.SetDT(workloads.cfl_dt(d.calcMinEdgeLength(), nodxelem=el.shape[1], factor=0.4))
    d.init()
    d.setField("v", v)
    return d


@pytest.mark.parametrize("separate", [False, True])
@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_renumbered_nodes(mesh, precision, separate):
    x, el = MESHES[mesh]()
    z = x[:, 2]
    v = np.zeros_like(x)
    v[:, 2] = -8.0 * (z - z.min()) / np.ptp(z)
    bottom, top = np.flatnonzero(z == z.min()), np.flatnonzero(z == z.max())
    new = np.random.default_rng(7).permutation(len(x))  # old node -> new node
    x2, v2 = np.empty_like(x), np.empty_like(v)
    x2[new], v2[new] = x, v
    a = make(x, el, bottom, top, v, precision)
    b = make(x2, new[el].astype(np.int32), new[bottom], new[top], v2, precision)
    for d in (a, b):
        if separate:
            d.timeFusedPhases(9)
        else:
            d.runFused(9, reaction=False)
    for name in ("x", "v", "u"):
        f, g = a.field(name).reshape(-1, 3), b.field(name).reshape(-1, 3)
        assert np.all(np.isfinite(f)) and np.any(f != (x if name == "x" else v))
        assert np.array_equal(f, g[new]), name
    for name in ("tau", "sigma", "pl_strain", "p"):
        assert np.array_equal(a.field(name), b.field(name)), name
