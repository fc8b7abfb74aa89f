"""Electrodes less than a rounding error's width off the centre of a myocardial cell, on a heart
whose voxels are all in classes.

The FP32 weight |e|^-3 is finite from 2^(-128/3) = 1.44e-13 voxels on.  Closer, the
lead is not finite, as on the centre itself; from there on it follows the FP64
oracle as far as its own sum can: it forms p . T + T3, whose two parts are
q / d times the result (q < 8 the electrode's place in a box of cells, d the
offset), each rounded to 2^-53, four operations: 4 x 8 x 2^-53 / d, doubled for
the two parts.
"""
import numpy as np
import pytest

from ekgsim_amd import synth as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def heart():
    from ekgsim_amd import Context, Heart
    ctx = Context(0)
    h = S.make_heart(24, seed=1)
    g = Heart(ctx, h.layer, h.seed)
    g.excite_delay(h.delay)
    g.set_tune(class_min=1)
    z, y, x = np.nonzero(h.layer > 0)
    i = np.argmin((z - 12) ** 2 + (y - 12) ** 2 + (x - 12) ** 2)
    yield h, g, O.excite_int(h.layer, h.seed, h.delay).astype(np.float64), np.array([z[i], y[i], x[i]], float) + 1.0
    g.close()
    ctx.close()


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("steps", [1, 4, 32, 64, 84, 120, 4096])
def test_close_electrode(heart, axis, steps):
    h, g, act, m = heart
    k = S.layer_k_from_params(S.random_params(3, 1, 11), 3)
    p = m.copy()
    p[axis] += steps * np.spacing(m[axis])  # exact
    d = p[axis] - m[axis]
    far = np.array([60.0, 50.0, 40.0])
    got = g.simulate(k, np.array([p, far]), "3D4", 0.0, 100.0, 1.0)
    alone = g.simulate(k, far[None], "3D4", 0.0, 100.0, 1.0)
    print(f"axis {axis}, offset {d:.3g}: {got[0, :3]}")
    assert np.array_equal(got[1], alone[0])
    if d < 2.0 ** (-128 / 3):
        assert not np.isfinite(got[0]).any()
        return
    ref = O.run(h.layer, act, k, p[None], "3D4", 0.0, 100.0, 1.0)[0]
    tol = 1e-5 + 2 * 4 * 8 * 2.0 ** -53 / d
    assert np.linalg.norm(got[0] - ref) <= tol * np.linalg.norm(ref)
