"""Paired passes (two kernels per step on small meshes) against the four
separate ones, bit for bit: `runFused` takes the paired passes there,
`timeFusedPhases` the separate ones.  Hexahedra and tetrahedra, both
precisions, every law class and option, odd and even run lengths, meshes of
one element, of several components and with nodes of more elements than one
register load holds, and a mesh with a node of no element (separate passes
only).
"""
import numpy as np
import pytest

from weldformfem_amd import WFX_FP32_MIXED, WFX_FP64, WFX_HOLLOMON, Domain, workloads

pytestmark = pytest.mark.gpu

STEEL = (200e9, 0.3, 7850.0)
JC = (300e6, 500e6, 0.3, 0.014, 1.0, 1.0, 1520.0, 20.0)
GMT = ((-2e-4, 0.15, 600e6, -1.5e-3, 1e-4, 0.01, -1e-5, 1e-4), (0.002, 3.0, 1e-3, 1e5, 20.0, 1200.0))


def fan(sectors, layers, tets=False, stray=False):
    """quadrilaterals around an axis, extruded: the axis nodes carry
    2 * sectors hexahedra (or their six tetrahedra each)"""
    a = 2 * np.pi * np.arange(2 * sectors) / (2 * sectors)
    ring = np.stack([np.cos(a), np.sin(a)], 1) * np.where(np.arange(2 * sectors) % 2, 1.0, 0.9)[:, None]
    plane = np.concatenate([np.zeros((1, 2)), ring]) * 0.1
    n2 = len(plane)
    x = np.concatenate([np.c_[plane, np.full(n2, 0.07 * k)] for k in range(layers + 1)])
    el = []
    for k in range(layers):
        for s in range(sectors):
            q = np.array([0, 1 + 2 * s, 2 + 2 * s, 1 + (2 * s + 2) % (2 * sectors)])
            el.append(np.r_[q + k * n2, q + (k + 1) * n2])
    el = np.array(el, dtype=np.int32)
    if tets:
        pat = np.array([[0, 1, 3, 5], [1, 2, 3, 5], [0, 5, 3, 4], [4, 5, 3, 7], [5, 6, 3, 7], [5, 2, 3, 6]])
        el = el[:, pat].reshape(-1, 4)
    if stray:
        x = np.r_[x, [[0.5, 0.5, 0.5]]]
    return x, np.ascontiguousarray(el), np.arange(n2), np.arange(layers * n2, (layers + 1) * n2)


def box(nx, ny, nz):
    x, el = workloads.hexa_box(nx, ny, nz, 0.05)
    return (x, el) + workloads.box_layers(nx, ny, nz)


def two_boxes():
    x, el, b, t = box(7, 6, 5)
    y, fl, c, u = box(3, 9, 4)
    y = y + [1.0, 0, 0]
    n = len(x)
    return np.r_[x, y], np.r_[el, fl + n].astype(np.int32), np.r_[b, c + n], np.r_[t, u + n]


MESHES = {
    "hexa1": lambda: box(1, 1, 1),
    "hexa9x8x7": lambda: box(9, 8, 7),
    "hexa17x16x15": lambda: box(17, 16, 15),
    "two boxes": two_boxes,
    "fan9": lambda: fan(9, 4),
    "fan15": lambda: fan(15, 3),
    "fan of tets": lambda: fan(5, 3, tets=True),
    "cylinder8": lambda: workloads.cylinder_tets(cells=8),
    "stray node": lambda: fan(6, 2, stray=True),
}


def make(mesh, precision, option):
    x, el, bottom, top = MESHES[mesh]()
    d = Domain(precision)
    d.CreateFromMesh(x, el, el.shape[1])
    d.setDensity(7850.0)
    if option in ("jc", "jc thermal cfl"):
        d.setMaterialJC(*STEEL, *JC)
    elif option == "gmt thermal":
        d.setMaterialGMT(*STEEL, 250e6, *GMT)
    elif option == "hollomon":
        d.setMaterial(WFX_HOLLOMON, *STEEL, 150e6, 600e6, 0.2)
    else:
        d.setMaterial(0, *STEEL, 1e4 if option == "yielding" else 100e6, 1e9, 0.0)
    for nd in bottom:
        d.AddBCVelNode(int(nd), 2, 0.0)
    for nd in top if option != "contact" else []:
        d.AddBCVelNode(int(nd), 2, -8.0)
    d.AddBCVelNode(int(bottom[0]), 0, 0.0)
    d.AllocateBCs()
    d.setReactionNodes(bottom)
    d.set("hg_coeff", 0.06)
    if "thermal" in option:
        d.setThermal(True, 50.0, 460.0, 0.9)
    if "expansion" in option:
        d.setThermalExpansion(1.2e-5)
    d.SetDT(workloads.cfl_dt(d.calcMinEdgeLength(), nodxelem=el.shape[1], factor=0.4))
    if "cfl" in option:
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
    return d


CASES = [(m, p, "plain", n) for m in MESHES for p in (WFX_FP64, WFX_FP32_MIXED) for n in (1, 2, 7, 12)]
CASES += [(m, p, o, 21) for m in ("hexa9x8x7", "cylinder8") for p in (WFX_FP64, WFX_FP32_MIXED)
          for o in ("yielding", "jc", "gmt thermal", "hollomon", "cfl", "jc thermal cfl", "thermal expansion")]
CASES += [("cylinder8", p, "contact", n) for p in (WFX_FP64, WFX_FP32_MIXED) for n in (20, 33)]


@pytest.mark.parametrize("mesh,precision,option,nsteps", CASES)
def test_equals_the_separate_passes(mesh, precision, option, nsteps):
    print(f"case: paired passes, {mesh}, precision {precision}, {option}, {nsteps} steps", flush=True)
    a, b = make(mesh, precision, option), make(mesh, precision, option)
    if mesh == "stray node":  # its division by a zero mass is reported, on both sides
        a.set("check_status", 0)
        b.set("check_status", 0)
    for n in (nsteps, 3):  # and a second run from the first one's state
        a.runFused(n)
        b.timeFusedPhases(n)
        for f in ("x", "u", "v", "a", "u_dt", "prev_a", "fi", "mdiag", "voln", "vol", "p", "tau", "eps", "sigma",
                  "pl_strain", "sigma_y", "T") + (("contforce", "cfn", "rigid_x") if option == "contact" else ()):
            np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
        if "cfl" in option:
            np.testing.assert_array_equal(a.dtHistory(n), b.dtHistory(n))
    if option == "yielding":
        assert np.all(a.field("pl_strain") > 0)
