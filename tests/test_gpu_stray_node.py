"""Meshes with a node of no element (accepted by the mesh calls; here held in
all directions): what such a node must not change."""
import numpy as np
import pytest

from weldformfem_amd import Domain, WFX_FP32_MIXED, WFX_FP64, workloads
from weldformfem_amd.adjoint import CompressionProblem

pytestmark = pytest.mark.gpu


def test_cfl_gradient():
    """The gradient with the per-step CFL time step is the one without the
    node.  The step length's cotangent is a sum over nodes and elements in an
    order the node shifts: some 300 roundings of 1e-16 a step and 60 steps, 2e-12
    of the largest term; the bar leaves 500 times that for cancellation."""
    print("case: per-step CFL adjoint with a node of no element", flush=True)
    n = 5
    x, el = workloads.hexa_box(n, n, n, 0.2)
    bottom, top = workloads.box_layers(n, n, n)
    grads = []
    for stray in (False, True):
        xs = np.r_[x.reshape(-1, 3), [[9.0, 9.0, 9.0]]] if stray else x
        pb = CompressionProblem(nsteps=60, every=9, mesh=(xs, el, 8, bottom, top), cfl=0.3)
        if stray:
            for d in range(3):
                pb.domain.AddBCVelNode(len(xs) - 1, d, 0.0)
            pb.domain.AllocateBCs()
        h = pb.forward([5e6, 1.1e9, 0.07])
        assert np.all(np.isfinite(h)) and np.any(h != 0)
        grads.append(np.asarray(pb.backward(1e-9 * h)))
    assert np.all(np.isfinite(grads[0])) and np.all(grads[0] != 0)
    np.testing.assert_allclose(grads[1], grads[0], rtol=1e-9)


@pytest.mark.parametrize("mesh", ["hexa", "tets"])  # nodal sums by a thread and by lanes
@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
def test_mass_with_varying_densities(precision, mesh):
    """The empty sum's mass, 0, and nothing but numbers in the other fields"""
    print(f"case: densities that vary, a node of no element, {mesh}, precision {precision}", flush=True)
    if mesh == "hexa":
        x, el = workloads.hexa_box(6, 5, 4, 0.05)
        bottom, top = workloads.box_layers(6, 5, 4)
    else:
        x, el, bottom, top = workloads.cylinder_tets(cells=8)
    x = np.r_[x.reshape(-1, 3), [[9.0, 9.0, 9.0]]]
    el = el.reshape(-1, 8 if mesh == "hexa" else 4)
    d = Domain(precision)
    d.CreateFromMesh(x, el, el.shape[1])
    for k in range(3):
        d.AddBCVelNode(len(x) - 1, k, 0.0)
    workloads.setup_compression(d, bottom, top, -1.0)
    d.init()
    d.setField("rho", 7000.0 + 8.0 * (np.arange(len(el)) % 97))
    d.runFused(5)
    m = d.field("mdiag")
    assert m[-1] == 0.0 and np.all(m[:-1] > 0)
    for f in ("x", "u", "v", "a", "fi", "tau", "p"):
        assert np.all(np.isfinite(d.field(f))), f
