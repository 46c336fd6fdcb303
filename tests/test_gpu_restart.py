"""wfx_init on a used domain gives the state of a new one, at odd sizes, in
both precisions, and the host's view of the densities follows them (uniform,
varying, and a density that is not positive).
"""
import numpy as np
import pytest

from weldformfem_amd import Domain, WFX_FP32_MIXED, WFX_FP64, workloads

pytestmark = pytest.mark.gpu

FIELDS = ("x", "v", "a", "u", "u_dt", "prev_a", "fi", "mdiag", "voln", "vol", "vol0", "rho", "p", "pl_strain",
          "sigma_y", "sigma", "tau", "eps", "strain_pl_incr", "f_hg", "detJ")


def make(precision, mesh):
    d = Domain(precision)
    x, el = workloads.hexa_box(*mesh, 0.1)
    bottom, top = workloads.box_layers(*mesh)
    d.CreateFromMesh(x, el, 8)
    workloads.setup_compression(d, bottom, top, -30.0, sy0=workloads.lognormal_sy0(el.shape[0], 1e6))
    d.init()
    return d, x


@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
@pytest.mark.parametrize("mesh", [(1, 1, 1), (5, 3, 1), (11, 7, 5), (40, 33, 31)])
def test_restart(precision, mesh):
    print(f"case: restart {mesh}, precision {precision}", flush=True)
    (a, x), (b, _) = make(precision, mesh), make(precision, mesh)
    a.runFused(5)
    a.run(2)
    a.setField("x", x)
    a.init()
    for f in FIELDS:
        np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
    np.testing.assert_array_equal(a.runFused(4), b.runFused(4))
    np.testing.assert_array_equal(a.field("u"), b.field("u"))


@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
def test_densities(precision):
    print(f"case: densities, precision {precision}", flush=True)
    d, _ = make(precision, (9, 8, 7))
    E = d.elem_count
    for rho in (np.full(E, 7000.0), np.linspace(6000.0, 9000.0, E), np.r_[np.full(E - 1, 7000.0), 6999.0]):
        d.setField("rho", rho)
        d.runFused(1, reaction=False)
        # the mass of every node: its elements' densities times their volumes' share
        el, vol = d.field("elnod").reshape(E, 8), d.field("vol")
        cnt, vn, rs = np.zeros(d.node_count), np.zeros(d.node_count), np.zeros(d.node_count)
        r = d.field("rho")
        for k in range(8):
            np.add.at(cnt, el[:, k], 1.0)
            np.add.at(vn, el[:, k], vol / 8)
            np.add.at(rs, el[:, k], r)
        np.testing.assert_allclose(d.field("mdiag"), vn * rs / cnt, rtol=1e-13)
