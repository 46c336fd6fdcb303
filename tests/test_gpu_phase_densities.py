"""Nodal masses of the separate phases after the densities changed and a run
was captured but not launched: phase 2 takes the present densities."""
import numpy as np
import pytest
import torch

from weldformfem_amd import Domain, WFX_FP32_MIXED, WFX_FP64, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before", ["init", "run"])
@pytest.mark.parametrize("mesh", ["hexa", "tets"])
@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
def test_phase_2_after_a_capture(precision, mesh, before):
    """m_i = V_i / n * (mean density of the node's elements): sums of at most 32
    terms, 3e-15 each, and the density's narrowing to float, here exact"""
    print(f"case: phase 2 after a capture, {mesh}, precision {precision}, after {before}", flush=True)
    d = Domain(precision)
    if mesh == "hexa":
        x, el = workloads.hexa_box(5, 4, 3, 0.05)
        bottom, top = workloads.box_layers(5, 4, 3)
    else:
        x, el, bottom, top = workloads.cylinder_tets(cells=6)
    n = el.shape[1]
    d.CreateFromMesh(x, el, n)
    workloads.setup_compression(d, bottom, top, -1.0)
    d.init()
    stream = torch.cuda.Stream()
    d.stream = stream.cuda_stream
    if before == "run":
        d.runFused(3)
    rho = 7000.0 + 8.0 * (np.arange(len(el)) % 97)
    d.setField("rho", rho)
    d.graphCapture(4)
    d.fusedPhase(1)
    d.fusedPhase(2)
    stream.synchronize()
    vol, N = d.field("vol"), len(x.reshape(-1, 3))
    total, mass, count = np.zeros(N), np.zeros(N), np.zeros(N)
    for a in range(n):
        np.add.at(total, el[:, a], vol)
        np.add.at(mass, el[:, a], rho)
        np.add.at(count, el[:, a], 1.0)
    np.testing.assert_allclose(d.field("mdiag"), total / n * mass / count, rtol=1e-14)
