"""Steps inside a run of per-step steps, whose nodal kernels and nodal sums are
merged, against the entry points called one by one and against runs of one
step each, bit for bit: both elements, both precisions, boundary values on
every component, external forces, thermal coupling, contact, the per-step CFL
time step, and a mesh without boundary conditions.
"""
import numpy as np
import pytest

from test_gpu_paired_passes import JC, STEEL, box
from weldformfem_amd import WFX_FP32_MIXED, WFX_FP64, Domain, workloads

pytestmark = pytest.mark.gpu

FIELDS = ("x", "u", "v", "a", "u_dt", "prev_a", "fi", "mdiag", "voln", "vol", "p", "tau", "eps", "sigma", "pl_strain",
          "sigma_y", "str_rate", "T")


def make(mesh, precision, option):
    x, el, bottom, top = box(9, 8, 7) if mesh == "hexa" else workloads.cylinder_tets(cells=6)
    d = Domain(precision)
    d.CreateFromMesh(x, el, el.shape[1])
    d.setDensity(7850.0)
    if option == "thermal":
        d.setMaterialJC(*STEEL, *JC)
    else:
        d.setMaterial(0, *STEEL, 100e6, 1e9, 0.0)
    if option != "free":
        for nd in bottom:
            d.AddBCVelNode(int(nd), 2, 0.0)
        for nd in top if option != "contact" else []:
            d.AddBCVelNode(int(nd), 2, -8.0)
        d.AddBCVelNode(int(bottom[0]), 0, 0.5)
        d.AddBCVelNode(int(bottom[1]), 1, -0.25)
        d.AddBCVelNode(int(bottom[1]), 1, 0.75)  # the last entry counts
    d.AllocateBCs()
    d.setReactionNodes(bottom)
    d.set("hg_coeff", 0.06)
    if option == "thermal":
        d.setThermal(True, 50.0, 460.0, 0.9)
        d.setThermalExpansion(1.2e-5)
    d.SetDT(workloads.cfl_dt(d.calcMinEdgeLength(), nodxelem=el.shape[1], factor=0.4))
    if option == "cfl":
        d.setCFL(0.2)
    if option == "contact":
        z = x[:, 2].max()
        die = np.array([[-3, -3, z], [3, -3, z], [-3, 3, z], [3, 3, z]], float)
        d.setRigidMesh(die, np.array([[0, 2, 1], [1, 2, 3]]), vel=[0.0, 0.0, -20.0])
        d.setContactParams(0.1, 0.2, 0.1)
    d.init()
    v = np.zeros_like(x)
    v[:, 2] = -8.0 * (x[:, 2] - x[:, 2].min()) / np.ptp(x[:, 2])
    d.setField("v", v)
    if option == "forces":
        d.setField("fe", 1e3 * np.sin(np.arange(3.0 * len(x))).reshape(-1, 3))
    return d


def equal(a, b):
    for f in FIELDS:
        np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)


def one_by_one(d):
    d.UpdatePrediction()
    for dim in range(3):
        d.ImposeBCV(dim)
    d.calcElemJAndDerivatives()
    d.CalcElemVol()
    d.CalcNodalVol()
    d.CalcNodalMassFromVol()
    d.calcElemStrainRates()
    d.calcElemPressure()
    d.CalcStressStrain(d.get("dt"))
    d.calcArtificialViscosity()
    d.calcElemForces()
    d.calcElemHourglassForces()
    d.assemblyForces()
    d.calcAccel()
    for dim in range(3):
        d.ImposeBCA(dim)
    d.UpdateCorrectionAccVel()
    for dim in range(3):
        d.ImposeBCV(dim)
    d.UpdateCorrectionPos()


@pytest.mark.parametrize("option", ["plain", "forces", "free"])
@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
@pytest.mark.parametrize("mesh", ["hexa", "tets"])
def test_run_equals_the_entry_points(mesh, precision, option):
    print(f"case: run against its entry points, {mesh}, precision {precision}, {option}", flush=True)
    a, b = make(mesh, precision, option), make(mesh, precision, option)
    for n in (1, 5):
        a.run(n)
        for _ in range(n):
            one_by_one(b)
        equal(a, b)


@pytest.mark.parametrize("option", ["plain", "thermal", "contact", "cfl"])
@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
def test_run_equals_single_steps(precision, option):
    print(f"case: run against single steps, precision {precision}, {option}", flush=True)
    a, b = make("tets", precision, option), make("tets", precision, option)
    h = np.asarray(a.run(12))
    hb = np.concatenate([np.asarray(b.run(1)).reshape(1, -1) for _ in range(12)])
    np.testing.assert_array_equal(h.reshape(12, -1), hb)
    equal(a, b)
