"""Hearts of many chunks (at least 512, from which a request that starts before the last activation is
reduced in eight parts, and more than 512 in a layer, from which a prefix block has 1,024 threads),
against the FP64 oracle: one lead count for every slot width and each edge of it, fewer and more
layers than parts, steps that end inside a tile, starts on either side of the last activation,
alone and in a batch (the same bits).  Tolerance: the framework's 1e-5 (relative L2).
"""
import numpy as np
import pytest

from ekgsim_amd import synth as S
from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module")
def hearts():
    from ekgsim_amd import Context, Heart
    ctx = Context(0)
    out = {}
    for layers in (1, 3, 12):
        h = S.make_heart(64, seed=5, n_layers=layers)
        T = S.layered_transfer(layers, layers + 2, 1.03, 1.57)
        g = Heart(ctx, h.layer, h.seed)
        g.excite_transfer(T)
        g.set_tune(chunk_voxels=64, class_min=-1)
        assert g.layout_info("3D4")["chunks"] >= 512
        act = O.excite_fp64(h.layer, h.seed, T)
        if layers == 1:
            assert np.count_nonzero(h.layer) > 512 * 64  # more than 512 chunks in the one layer
        out[layers] = (h, g, act)
    yield out
    for _, g, _ in out.values():
        g.close()
    ctx.close()


@pytest.mark.parametrize("layers", [1, 3, 12])
@pytest.mark.parametrize("leads", [1, 4, 5, 12, 16])
@pytest.mark.parametrize("when", ["before", "inside", "last", "after"])
def test_many_chunks(hearts, layers, leads, when):
    h, g, act = hearts[layers]
    last = float(act[h.layer > 0].max())
    start = {"before": 0.0, "inside": round(last / 2), "last": last - 1.0, "after": last}[when]
    x = S.random_params(layers, leads, 70 + leads)
    k = S.layer_k_from_params(x, layers)
    pos = S.lead_positions(64, leads)
    steps = 61 if when == "before" else 43  # neither a multiple of the tile's 8 steps
    ref = O.run(h.layer, act, k, pos, "3D4", start, float(steps), 1.0)
    got = g.simulate(k, pos, "3D4", start, float(steps), 1.0)
    err = rel_l2(got, ref)
    print(f"{layers} layers, {leads} leads, start {start} ({when}): rel-L2 {err:.2e}")
    assert got.shape == (leads, steps)
    assert err <= TOL
    batch = g.simulate_batch(np.stack([k, k, k]), np.stack([pos, pos, pos]), "3D4", start, float(steps), 1.0)
    for b in range(3):
        assert np.array_equal(batch[b], got)
