"""Field transfers around the chunk size of the pinned ring (524,288 values):
what is set is read back bit for bit, in the caller's element order, for
nodal and element fields, one to six components, both precisions (floats
keep their rounding), and the spin's zero diagonal stays zero.
"""
import numpy as np
import pytest

from weldformfem_amd import Domain, WFX_FP32_MIXED, WFX_FP64, workloads

pytestmark = pytest.mark.gpu

# elements and values on both sides of one chunk, of the ring (16 chunks), and odd sizes
MESHES = [(1, 1, 1), (7, 5, 3), (43, 32, 31), (64, 64, 128), (113, 112, 111)]


@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
@pytest.mark.parametrize("mesh", MESHES)
def test_set_then_get(precision, mesh):
    print(f"case: field transfer {mesh}, precision {precision}", flush=True)
    d = Domain(precision)
    x, el = workloads.hexa_box(*mesh, 0.1)
    d.CreateFromMesh(x, el, 8)
    np.testing.assert_array_equal(d.field("x"), x.reshape(-1))
    rng = np.random.default_rng(3)
    real = np.float64 if precision == WFX_FP64 else np.float32
    E, N = el.shape[0], x.shape[0]
    for name, size, t in [("v", 3 * N, np.float64), ("tau", 6 * E, real), ("pl_strain", E, real),
                          ("T", N, np.float64)]:
        a = rng.standard_normal(size)
        d.setField(name, a)
        np.testing.assert_array_equal(d.field(name), a.astype(t).astype(np.float64))
    w = rng.standard_normal((E, 6))
    d.setField("rot_rate", w)
    w[:, :3] = 0.0
    np.testing.assert_array_equal(d.field("rot_rate").reshape(E, 6), w.astype(real).astype(np.float64))
