"""Field transfers around the lines between the copies on the host and the
kernels (16 and 64 KiB on the device, 4500 items): values of known position
come out in the caller's order, and what is set goes where the kernels read it.
"""
import numpy as np
import pytest

from weldformfem_amd import Domain, WFX_FP32_MIXED, WFX_FP64, workloads

pytestmark = pytest.mark.gpu

# elements: scalars of 1331 to 6859 items, 5 KB to 55 KB; tensors of six times that
MESHES = [(11, 11, 11), (13, 13, 13), (16, 16, 16), (17, 16, 16), (17, 16, 17), (19, 19, 19)]


@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
@pytest.mark.parametrize("mesh", MESHES)
def test_element_order(precision, mesh):
    print(f"case: small fields, {mesh}, precision {precision}", flush=True)
    real = np.float64 if precision == WFX_FP64 else np.float32
    x, el = workloads.hexa_box(*mesh, 1.0)
    x = x.reshape(-1, 3)
    x = 0.05 * (x + 0.01 * x * x * [1.0, 0.9, 0.8])  # cells of unequal edges
    d = Domain(precision)
    d.CreateFromMesh(x, el, 8)
    bottom, top = workloads.box_layers(*mesh)
    workloads.setup_compression(d, bottom, top, -1.0)
    d.init()
    np.testing.assert_array_equal(d.field("x"), x.reshape(-1))
    # read: volumes the kernels formed (products of the edges; FP32-mixed from
    # float differences, some 30 roundings of 6e-8)
    vol = np.prod(x[el[:, 6]] - x[el[:, 0]], axis=1)
    np.testing.assert_allclose(d.field("vol"), vol, rtol=1e-13 if precision == WFX_FP64 else 4e-6)
    # set: densities the kernels read into the masses
    E = len(el)
    rho = 7000.0 + 8.0 * (np.arange(E) % 97)
    d.setField("rho", rho)
    d.fusedPhase(1)
    d.fusedPhase(2)
    total, mass = np.zeros(len(x)), np.zeros(len(x))
    v = d.field("vol")
    for a in range(8):
        np.add.at(total, el[:, a], v)
        np.add.at(mass, el[:, a], rho)
    np.testing.assert_allclose(d.field("mdiag"), total / 8 * mass / np.bincount(el.ravel()), rtol=1e-14)
    # back and forth
    rng = np.random.default_rng(5)
    for name, size, t in (("v", x.size, np.float64), ("T", len(x), np.float64), ("pl_strain", E, real),
                          ("tau", 6 * E, real)):
        a = rng.standard_normal(size)
        d.setField(name, a)
        np.testing.assert_array_equal(d.field(name), a.astype(t).astype(np.float64))
    w = rng.standard_normal((E, 6))
    d.step()  # a per-step step: its intermediates can be read
    d.setField("rot_rate", w)
    w[:, :3] = 0.0
    np.testing.assert_array_equal(d.field("rot_rate").reshape(E, 6), w.astype(real).astype(np.float64))
