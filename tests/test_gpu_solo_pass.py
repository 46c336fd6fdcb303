"""Solo pass (all steps of a run but the last in one launch, for FP64 meshes
whose clusters share no node) against the four separate passes, bit for bit:
one element up to a full cluster, tetrahedra around a crowded axis, several
components, every law class, external forces, runs longer than a launch, a
second run from the first one's state; its reaction record against the last
steps of shorter runs; and a captured run against an eager one.
"""
import numpy as np
import pytest
import torch

from test_gpu_paired_passes import GMT, JC, STEEL, box, fan
from weldformfem_amd import WFX_FP64, WFX_HOLLOMON, Domain, workloads

pytestmark = pytest.mark.gpu

FIELDS = ("x", "u", "v", "a", "u_dt", "prev_a", "fi", "mdiag", "voln", "vol", "p", "tau", "eps", "sigma", "pl_strain",
          "sigma_y")


def three_boxes():
    parts, n = [], 0
    for k, size in enumerate([(5, 4, 3), (1, 1, 1), (4, 8, 8)]):
        x, el, b, t = box(*size)
        parts.append((x + [2.0 * k, 0, 0], el + n, b + n, t + n))
        n += len(x)
    return tuple(np.concatenate([p[i] for p in parts]) for i in range(3)) + (np.concatenate([p[3] for p in parts]),)


MESHES = {
    "hexa1": lambda: box(1, 1, 1),
    "hexa6x6x6": lambda: box(6, 6, 6),
    "full cluster": lambda: box(16, 4, 4),
    "fan of tets": lambda: fan(5, 3, tets=True),
    "fan15": lambda: fan(15, 3),
    "three boxes": three_boxes,
}


def make(mesh, option):
    x, el, bottom, top = MESHES[mesh]()
    d = Domain(WFX_FP64)
    d.CreateFromMesh(x, el.astype(np.int32), el.shape[1])
    d.setDensity(7850.0)
    if option == "jc":
        d.setMaterialJC(*STEEL, *JC)
    elif option == "gmt":
        d.setMaterialGMT(*STEEL, 250e6, *GMT)
    elif option == "hollomon":
        d.setMaterial(WFX_HOLLOMON, *STEEL, 150e6, 600e6, 0.2)
    else:
        d.setMaterial(0, *STEEL, 1e4 if option == "yielding" else 100e6, 1e9, 0.0)
    for nd in bottom:
        d.AddBCVelNode(int(nd), 2, 0.0)
    for nd in top:
        d.AddBCVelNode(int(nd), 2, -8.0)
    d.AddBCVelNode(int(bottom[0]), 0, 0.0)
    d.AllocateBCs()
    d.setReactionNodes(bottom)
    d.set("hg_coeff", 0.06)
    d.SetDT(workloads.cfl_dt(d.calcMinEdgeLength(), nodxelem=el.shape[1], factor=0.4))
    d.init()
    v = np.zeros_like(x)
    v[:, 2] = -8.0 * (x[:, 2] - x[:, 2].min()) / np.ptp(x[:, 2])
    d.setField("v", v)
    if option == "forces":
        d.setField("fe", 1e3 * np.sin(np.arange(3.0 * len(x))).reshape(-1, 3))
    return d


CASES = [(m, "plain", n) for m in MESHES for n in (2, 3, 13)]
CASES += [("hexa6x6x6", o, 14) for o in ("yielding", "jc", "gmt", "hollomon", "forces")]
CASES += [("fan of tets", o, 14) for o in ("yielding", "jc", "gmt", "hollomon", "forces")]
CASES += [("hexa1", "plain", n) for n in (513, 514, 1030)]


@pytest.mark.parametrize("mesh,option,nsteps", CASES)
def test_equals_the_separate_passes(mesh, option, nsteps):
    print(f"case: solo pass, {mesh}, {option}, {nsteps} steps", flush=True)
    a, b = make(mesh, option), make(mesh, option)
    for n in (nsteps, 4):
        a.runFused(n)
        b.timeFusedPhases(n)
        for f in FIELDS:
            np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
    if option == "yielding":
        assert np.all(a.field("pl_strain") > 0)


@pytest.mark.parametrize("mesh,nsteps", [("hexa1", 700), ("hexa6x6x6", 20), ("three boxes", 20), ("fan of tets", 20)])
def test_reaction_record(mesh, nsteps):
    print(f"case: solo pass, reactions, {mesh}, {nsteps} steps", flush=True)
    h = np.asarray(make(mesh, "plain").runFused(nsteps)).reshape(nsteps, -1)
    assert np.all(np.isfinite(h)) and np.any(h != 0)
    for k in sorted({1, 2, nsteps // 2, min(511, nsteps - 2), min(512, nsteps - 1), nsteps - 1}):
        # the last step of a run takes the node pass of the separate passes
        s = np.asarray(make(mesh, "plain").runFused(k + 1)).reshape(k + 1, -1)
        np.testing.assert_array_equal(h[:k + 1], s)


@pytest.mark.parametrize("mesh", ["hexa1", "three boxes"])
def test_captured(mesh):
    print(f"case: solo pass, captured, {mesh}", flush=True)
    a, b = make(mesh, "plain"), make(mesh, "plain")
    stream = torch.cuda.Stream()
    a.stream = stream.cuda_stream
    a.graphCapture(30)
    for _ in range(3):
        np.testing.assert_array_equal(a.graphLaunch(), b.runFused(30))
        for f in FIELDS:
            np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
