"""The reaction record of a run: rows kept in a ring of 512 steps and summed
once per filled ring.  The last entry of a history equals the reaction of the
state the run leaves, bit for bit, at run lengths around the ring's size; the
per-step path's history equals stepping one by one.  Groups share nodes, list
a node twice, and one is empty.
"""
import numpy as np
import pytest

from weldformfem_amd import Domain, WFX_FP32_MIXED, WFX_FP64, workloads

pytestmark = pytest.mark.gpu


def make(precision):
    d = Domain(precision)
    x, el = workloads.hexa_box(5, 4, 3, 0.1)
    bottom, top = workloads.box_layers(5, 4, 3)
    d.CreateFromMesh(x, el, 8)
    dt = workloads.setup_compression(d, bottom, top, -1.0)
    d.SetDT(0.2 * dt)
    d.setReactionGroups([top, bottom[:7], np.r_[top[3:5], bottom[2:4], top[3:4]], np.zeros(0, int), np.r_[119, 0, 64, 63]])
    d.init()
    return d


@pytest.mark.parametrize("precision", [WFX_FP64, WFX_FP32_MIXED])
@pytest.mark.parametrize("nsteps", [1, 511, 512, 513, 1030])
def test_fused_history_ends_at_the_state(precision, nsteps):
    print(f"case: fused reaction record, precision {precision}, {nsteps} steps", flush=True)
    d = make(precision)
    h = d.runFused(nsteps)
    assert h.shape == (nsteps, 5) and np.all(np.isfinite(h))
    np.testing.assert_array_equal(h[-1], d.reactionForce())
    assert np.all(h[:, 3] == 0.0) and np.all(h[:, 0] != 0.0)


def test_per_step_history_equals_single_steps():
    print("case: per-step reaction record, 520 steps", flush=True)
    a, b = make(WFX_FP64), make(WFX_FP64)
    h = a.run(520)
    for k in range(520):
        b.step()
        np.testing.assert_array_equal(h[k], b.reactionForce())
