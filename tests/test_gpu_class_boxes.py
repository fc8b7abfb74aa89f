"""The class-box kernel (activation classes summed on the int8 matrix cores)
where its scales, passes and tiles can go wrong, against the FP64 oracle:

* electrodes at every distance its weight scales distinguish: far outside the grid, some
  voxels off the heart, on and near the centres of empty cells inside it, and
  fractions of a voxel from the centre of a myocardial cell (the passes
  over the weights' fractions), all in one 16-lead row;
* an electrode on the centre of a myocardial cell, whose weight is infinite: that
  lead is not finite and the others keep their bits;
* conduction-matrix hearts with every voxel in a class (more classes in a box
  than one listing holds, regions cut by their class count);
* lead counts that leave rows of 16 partly filled, alone and across requests.

Tolerance: the framework's 1e-5 per lead (relative L2); the FP32 weights alone
account for about 6e-8 of it.
"""
import numpy as np
import pytest

from ekgsim_amd import synth as S
from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module")
def mfma():
    from ekgsim_amd import Context
    c = Context(0)
    yield c
    c.close()


def _heart(ctx, n, seed):
    from ekgsim_amd import Heart
    h = S.make_heart(n, seed=seed)
    g = Heart(ctx, h.layer, h.seed)
    g.excite_delay(h.delay)
    return h, g, O.excite_int(h.layer, h.seed, h.delay).astype(np.float64)


def _k(n_layers=3, seed=11):
    return S.layer_k_from_params(S.random_params(n_layers, 1, seed), n_layers)


def _centre(h, myo):
    """Coordinate + 1 of a cell near the grid's middle that is (not) myocardial."""
    z, y, x = np.nonzero((h.layer > 0) == myo)
    n = np.array(h.layer.shape) / 2.0
    i = np.argmin((z - n[0]) ** 2 + (y - n[1]) ** 2 + (x - n[2]) ** 2)
    return np.array([z[i], y[i], x[i]], float) + 1.0


@pytest.mark.parametrize("nhood", ["3D4", "3D8"])
def test_electrode_distances(mfma, nhood):
    h, g, act = _heart(mfma, 24, 3)
    m, e = _centre(h, True), _centre(h, False)
    pos = np.array([
        [1.0e4, -3.0e3, 2.0e3], [300.0, 12.0, 12.0], [40.0, 30.0, 12.0], [33.5, 12.0, 12.0], [12.0, 28.2, 12.0],
        e, e + [1e-3, 0, 0], e + [0.25, -0.4, 0.1],
        m + [0.5, 0.5, 0.5], m + [0.3, -0.2, 0.4], m + [0.05, 0, 0], m + [0, 0.01, 0], m + [1e-3, 1e-3, 0],
        [1.0, 1.0, 1.0], [24.0, 24.0, 24.0], m + [3.2, 0.1, 0.0]])
    assert pos.shape == (16, 3)
    ref = O.run(h.layer, act, _k(), pos, nhood, 0.0, 200.0, 1.0)
    got = g.simulate(_k(), pos, nhood, 0.0, 200.0, 1.0)
    for i in range(16):
        err = rel_l2(got[i], ref[i])
        print(f"{nhood} electrode {pos[i]}: rel-L2 {err:.2e}")
        assert err <= TOL, i
    g.close()


def test_electrode_on_a_cell_centre(mfma):
    h, g, act = _heart(mfma, 24, 3)
    good = S.lead_positions(24, 6)
    bad = good.copy()
    bad[2] = _centre(h, True)
    a = g.simulate(_k(), good, "3D4", 0.0, 200.0, 1.0)
    b = g.simulate(_k(), bad, "3D4", 0.0, 200.0, 1.0)
    assert not np.all(np.isfinite(b[2]))
    for i in (0, 1, 3, 4, 5):
        assert np.array_equal(a[i], b[i]), i
    g.close()


@pytest.mark.parametrize("nhood", ["3D4", "3D8"])
def test_every_voxel_its_own_class(mfma, nhood):
    from ekgsim_amd import Heart
    h = S.make_heart(20, seed=4)
    T = S.layered_transfer(3, 5, 1.07, 1.63)
    act = O.excite_fp64(h.layer, h.seed, T)
    g = Heart(mfma, h.layer, h.seed)
    g.excite_transfer(T)
    g.set_tune(class_min=1)
    info = g.layout_info(nhood)
    print(info)
    assert info["class_voxels"] == info["voxels"] and info["classes"] > 300
    pos = S.lead_positions(20, 5)
    ref = O.run(h.layer, act, _k(), pos, nhood, 0.0, 200.0, 1.0)
    assert rel_l2(g.simulate(_k(), pos, nhood, 0.0, 200.0, 1.0), ref) <= TOL
    g.close()


@pytest.mark.parametrize("leads", [(1,), (16, 16, 16), (3, 5, 2, 7), (15, 1, 2), (12,) * 9])
def test_rows_across_requests(mfma, leads):
    h, g, act = _heart(mfma, 26, 6)
    reqs = []
    for r, L in enumerate(leads):
        x = S.random_params(3, L, 900 + r)
        reqs.append((S.layer_k_from_params(x, 3), S.move_leads(S.lead_positions(26, L), S.displacements(x, 3, L)),
                     0.0, 150.0, 1.0))
    got = g.simulate_many(reqs, "3D4")
    for r, (k, p, st, ln, dt) in enumerate(reqs):
        assert rel_l2(got[r], O.run(h.layer, act, k, p, "3D4", st, ln, dt)) <= TOL, r
        # LP differs between the group and a lone request, the sums do not
        alone = g.simulate(k, p, "3D4", st, ln, dt)
        assert rel_l2(got[r], alone) <= 1e-13, r
    g.close()
