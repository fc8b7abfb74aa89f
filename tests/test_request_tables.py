"""The request descriptors handed to the library: table and single form against
each request's own arrays, for every order, stride, type and count the entry
points take.
"""
import ctypes as C

import numpy as np
import pytest

from ekgsim_amd import _capi as A


def _read(s):
    k = np.ctypeslib.as_array(s.layer_k, shape=(s.n_layers, 9)).copy() if s.n_layers else np.zeros((0, 9))
    p = np.ctypeslib.as_array(s.lead_pos, shape=(s.n_leads, 3)).copy() if s.n_leads else np.zeros((0, 3))
    return k, p, s.nhood, s.start, s.length, s.dt


def _same(s, k, p, nhood, start, length, dt):
    gk, gp, *rest = _read(s)
    assert np.array_equal(gk, np.asarray(k, np.float64).reshape(-1, 9))
    assert np.array_equal(gp, np.asarray(p, np.float64).reshape(-1, 3))
    assert rest == [A.NHOOD[nhood] if isinstance(nhood, str) else nhood, start, length, dt]


def _forms(a):
    yield a
    yield np.asfortranarray(a)
    yield a.astype(np.float32)
    yield np.repeat(a, 2, axis=0)[::2]
    yield a[::-1]
    r = a.copy()
    r.flags.writeable = False
    yield r


@pytest.mark.parametrize("batch,layers,leads", [(0, 3, 2), (1, 1, 1), (5, 24, 16), (3, 0, 2), (3, 2, 0)])
def test_uniform_table(batch, layers, leads):
    rng = np.random.default_rng(batch + layers)
    for k in _forms(rng.random((batch, layers, 9))):
        for p in _forms(rng.random((batch + 1, leads, 3))):
            k64, p64 = np.asarray(k, np.float64), np.asarray(p, np.float64)
            d = A._Descs.uniform(k64, p64, "3D8", 1.5, 300.0, 0.25)
            assert len(d.s) == batch
            for b in range(batch):
                _same(d.s[b], k64[b], p64[b], "3D8", 1.5, 300.0, 0.25)
    flat = rng.random((batch, 9 * layers))
    if batch and layers:
        d = A._Descs.uniform(flat, rng.random((batch, leads, 3)), 2, 0.0, 1.0, 1.0)
        _same(d.s[batch - 1], flat[batch - 1], np.asarray(_read(d.s[batch - 1])[1]), 2, 0.0, 1.0, 1.0)


def test_refused_shapes():
    k, p = np.zeros((3, 2, 9)), np.zeros((3, 4, 3))
    with pytest.raises(IndexError):
        A._Descs.uniform(k, p[:2], "3D4", 0.0, 1.0, 1.0)
    with pytest.raises(ValueError):
        A._Descs.uniform(np.zeros((3, 2, 8)), p, "3D4", 0.0, 1.0, 1.0)
    with pytest.raises(ValueError):
        A._Descs.uniform(k, np.zeros((3, 4, 2)), "3D4", 0.0, 1.0, 1.0)
    with pytest.raises(KeyError):
        A._Descs.uniform(k, p, "4D", 0.0, 1.0, 1.0)


def test_mixed_table_and_single():
    rng = np.random.default_rng(4)
    reqs = []
    for i, (k, p) in enumerate(zip(_forms(rng.random((3, 9))), _forms(rng.random((4, 3))))):
        reqs.append((k[:1 + i % 3], p[:i % 5], float(i), 100.0 + i, 0.5))
    reqs.append(([[1.0] * 9], [[1, 2, 3]], 0.0, 1.0, 1.0))
    ks, ps, st, ln, dt = zip(*reqs)
    d = A._Descs(ks, ps, "2D4", st, ln, dt)
    assert C.sizeof(d.s) == len(reqs) * C.sizeof(A.SimDesc)
    for s, (k, p, start, length, step) in zip(d.s, reqs):
        _same(s, k, p, "2D4", start, length, step)
        _same(A._Desc(k, p, "2D4", start, length, step).s, k, p, "2D4", start, length, step)
