"""Hearts with so many classes to a box that the waves of a class-box block divide them into two or four
parts, against the FP64 oracle: parts of unequal size, boxes with more classes than one
listing holds, lead rows partly filled, an electrode near a cell and one on its
centre; alone, in a batch, and in one group with hearts cut otherwise (the same bits).  Tolerance: the framework's 1e-5
per lead (relative L2).
"""
import numpy as np
import pytest

from ekgsim_amd import synth as S
from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-5

# grid, layers, class_min: 19, 49, 62 and 90 classes a box on average (1, 2, 4 and 4 parts)
HEARTS = [(40, 3, 8), (48, 9, 8), (48, 12, 4), (40, 24, 1)]


@pytest.fixture(scope="module", params=HEARTS, ids=lambda p: "%d^3-%d-layers" % p[:2])
def heart(request):
    from ekgsim_amd import Context, Heart
    n, layers, class_min = request.param
    ctx = Context(0)
    h = S.make_heart(n, seed=4, n_layers=layers)
    g = Heart(ctx, h.layer, h.seed)
    g.excite_delay(h.delay)
    g.set_tune(class_min=class_min)
    yield n, layers, h, g, O.excite_int(h.layer, h.seed, h.delay).astype(np.float64)
    g.close()
    ctx.close()


@pytest.mark.parametrize("nhood", ["3D4", "3D8"])
@pytest.mark.parametrize("leads", [1, 6, 16])
def test_many_classes(heart, leads, nhood):
    n, layers, h, g, act = heart
    k = S.layer_k_from_params(S.random_params(layers, 1, 21), layers)
    pos = S.lead_positions(n, leads)
    z, y, x = np.nonzero(h.layer > 0)
    cell = np.array([z[len(z) // 2], y[len(z) // 2], x[len(z) // 2]], float) + 1.0
    pos[0] = cell + [0.3, -0.2, 0.1]
    got = g.simulate(k, pos, nhood, 0.0, 120.0, 1.0)
    ref = O.run(h.layer, act, k, pos, nhood, 0.0, 120.0, 1.0)
    err = max(rel_l2(got[i], ref[i]) for i in range(leads))
    print(f"{n}^3, {layers} layers, {leads} leads, {nhood}: {g.layout_info(nhood)['classes']} classes, rel-L2 {err:.2e}")
    assert err <= TOL
    other = np.tile(pos[-1:], (leads, 1))
    other[0] = cell  # not finite; the other requests' leads of its row keep their bits
    batch = g.simulate_batch(np.stack([k, k, k]), np.stack([pos, other, pos]), nhood, 0.0, 120.0, 1.0)
    assert not np.isfinite(batch[1][0]).any()
    assert np.array_equal(batch[0], got) and np.array_equal(batch[2], got)


def test_hearts_of_every_cut_in_one_group():
    from ekgsim_amd import Context, Heart, Server
    ctx = Context(0)
    hearts = []
    for n, layers, class_min in HEARTS:
        h = S.make_heart(n, seed=4, n_layers=layers)
        g = Heart(ctx, h.layer, h.seed)
        g.excite_delay(h.delay)
        g.set_tune(class_min=class_min)
        hearts.append((n, layers, g))
    srv = Server(ctx, n_streams=1)
    ids = [srv.add_heart(g) for _, _, g in hearts]
    reqs = []
    for q in range(40):  # interleaved: the server orders a group by heart
        n, layers, g = hearts[q % 4]
        k = S.layer_k_from_params(S.random_params(layers, 1, 60 + q), layers)
        reqs.append((q % 4, k, S.lead_positions(n, 9 + q % 4)))
    tickets = [srv.submit(ids[i], k, p, "3D4", 0.0, 80.0, 1.0) for i, k, p in reqs]
    got = [srv.wait(t)[0] for t in tickets]
    print(f"{srv.stats()['groups']} groups")
    assert srv.stats()["groups"] < len(reqs)
    for (i, k, p), e in zip(reqs, got):
        assert np.array_equal(e, hearts[i][2].simulate(k, p, "3D4", 0.0, 80.0, 1.0))
    srv.close()
    for _, _, g in hearts:
        g.close()
    ctx.close()
