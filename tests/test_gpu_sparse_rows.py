"""Sparse FP32 steps look up the sites across a row's end once per row: rows
of 1 and 2 sites (both neighbours across the end), rows that end inside, at
and beyond a 32-site word of the rank index, in both models and both
dimensions, bit for bit against the dense layout, and a batch of such crops
against the single domains."""
import numpy as np
import pytest

from lbflow_amd import cases as CS

pytestmark = pytest.mark.gpu

SHAPES = [(5, 13, 1), (7, 6, 2), (4, 5, 3), (3, 9, 32), (4, 7, 33), (2, 3, 64), (1, 17, 31), (1, 5, 1)]


def _labels(shape, phi=0.7):
    rng = np.random.default_rng(sum(shape))
    g = np.where(rng.random(shape) < phi, np.where(rng.random(shape) < 0.5, 75, 76), 255)
    return g.astype(np.uint8)


def _spec(shape, model):
    labels = [CS.label_line(75, 'GV', 1e-5, 1, 0), CS.label_line(76, 'VD', phase=1 if model == 'color' else 0),
              CS.label_line(255, 'SD', 60)]
    kw = dict(sigma=1e-3, beta=0.7, tau=(0.9, 0.7)) if model == 'color' else dict(tau=(0.8,))
    return CS.make('rows', _labels(shape), labels, model=model, eq='MRT', **kw)


@pytest.mark.parametrize('model', ['scsp', 'color'])
@pytest.mark.parametrize('shape', SHAPES, ids=lambda s: 'x'.join(map(str, s)))
def test_sparse_equals_dense(shape, model):
    from lbflow_amd.engine import FP32, Engine
    spec = _spec(shape, model)
    pops = []
    for dense in (False, True):
        e = Engine(CS.lattice(spec), CS.geometry(spec), FP32, False, dense).init()
        e.advance(12)
        pops.append(e.populations())
    keep = np.tile(CS.geometry(spec) != 255, pops[0].size // CS.geometry(spec).size)
    assert np.isfinite(pops[0][keep]).all()
    assert np.array_equal(pops[0][keep], pops[1][keep])


def test_batch_equals_single_domains():
    from lbflow_amd.engine import FP32, Batch, Engine
    crops = [np.where(_labels(s) == 255, 255, 75).astype(np.uint8) for s in SHAPES if s[0] > 1]
    labels = {75: ('GV', 1e-5, 1, 0), 255: ('SD', 90.0, 0, 0)}
    b = Batch(3, 19, 'MRT', 0.8, 1.0, labels, crops)
    b.init().advance(12)
    for c, g in enumerate(crops):
        case = dict(D=3, Q=19, size=g.shape, model='scsp', eq='MRT', tau=(0.8,), density=(1.0,), labels=labels)
        e = Engine(case, g, FP32, stream_solids=False).init()
        e.advance(12)
        assert np.array_equal(b.populations(c), e.populations())
