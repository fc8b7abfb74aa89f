"""Hearts of few and many activation classes and of nothing but classes,
against the FP64 oracle: fewer classes than the class ECG kernel's waves and
one more than a multiple, several layers within one wave's share, steps around
its blocks of 64, lead counts around the slot widths.  Tolerance: the
framework's 1e-5 (relative L2).  A heart that is one class as a whole has no
potential at all (every cell's dipoles cancel): there the oracle returns its
rounding noise, and the bound is absolute, 1e-9 beside the thousands of the others.
"""
import numpy as np
import pytest

from ekgsim_amd import synth as S
from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module")
def ctx():
    from ekgsim_amd import Context
    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("leads,length", [(1, 63.0), (4, 64.0), (5, 65.0), (12, 1.0), (16, 129.0)])
@pytest.mark.parametrize("classes", [1, 7, 8, 9, 33])
def test_class_counts(ctx, classes, leads, length):
    from ekgsim_amd import Heart
    n, layers = 24, min(classes, 5)
    z = np.arange(n)[:, None, None] + np.zeros((n, n, n), int)
    # slabs of one time each; a layer holds whole slabs
    slab = z * classes // n if classes <= n else (np.arange(n ** 3).reshape(n, n, n) * classes) // n ** 3
    layer = (1 + slab * layers // classes).astype(np.uint8)
    act = 1.0 + 1.75 * slab.astype(np.float64)
    g = Heart(ctx, layer)
    g.set_activation(act)
    assert g.layout_info()["classes"] == classes
    k = S.layer_k_from_params(S.random_params(layers, leads, 60 + classes), layers)
    pos = S.lead_positions(n, leads)
    got = g.simulate(k, pos, "3D4", 10.0, length, 1.0)
    ref = O.run(layer, act, k, pos, "3D4", 10.0, length, 1.0)
    err = np.abs(got - ref).max() if classes == 1 else rel_l2(got, ref)
    print(f"{classes} classes, {leads} leads, {length} ms: error {err:.2e}")
    assert err <= (1e-9 if classes == 1 else TOL)
    batch = g.simulate_batch(np.stack([k] * 3), np.stack([pos] * 3), "3D4", 10.0, length, 1.0)
    assert all(np.array_equal(b, got) for b in batch)
    g.close()
