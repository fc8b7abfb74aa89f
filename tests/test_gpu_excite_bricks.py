"""The excitation sweep against the oracle, bit for bit: grids one voxel short
of, at and past the 8-voxel bricks, flat grids, empty voxels inside and between
bricks, unreached islands, seeds on brick faces, zero lags, and a conduction
matrix whose row of the empty layer holds no number.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from ekgsim_amd import Context
    c = Context(0)
    yield c
    c.close()


def _grid(shape, layers, fill, seed):
    rng = np.random.default_rng(seed)
    layer = np.where(rng.random(shape) < fill, rng.integers(1, layers + 1, shape), 0).astype(np.uint8)
    start = np.zeros(shape, np.uint8)
    for z, y, x in ((0, 0, 0), (shape[0] - 1, shape[1] // 2, min(7, shape[2] - 1)), (shape[0] // 2, min(8, shape[1] - 1), 0)):
        layer[z, y, x] = 1
        start[z, y, x] = 1
    return rng, layer, start


@pytest.mark.parametrize("fill", [0.25, 0.7, 1.0])
@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 8, 9), (8, 8, 8), (1, 16, 17), (9, 1, 24), (17, 23, 15), (33, 16, 8)])
def test_excite_bitwise(ctx, shape, fill):
    from ekgsim_amd import Heart
    rng, layer, start = _grid(shape, 4, fill, sum(shape))
    T = rng.uniform(0.0, 3.0, (6, 5))
    T[1, 1] = 0.0
    T[0, :] = np.nan  # the empty layer: never used
    h = Heart(ctx, layer, start)
    h.excite_transfer(T)
    ref = O.excite_fp64(layer, start, np.nan_to_num(T))
    assert np.array_equal(h.activation().view(np.uint64), ref.view(np.uint64))
    delay = rng.integers(0, 4, shape).astype(np.uint8)
    h.excite_delay(delay)
    assert np.array_equal(h.activation(), O.excite_int(layer, start, delay).astype(np.float64))
    h.close()
