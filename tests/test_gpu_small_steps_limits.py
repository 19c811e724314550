"""FP64 steps several to a launch, where their rules end: two-phase work orders
whose padded entries just fill or just miss the limit (the count is asserted,
so that each case runs the kernel it is there for), per-site relaxation times
in D3Q19, more steps than one launch holds; and single-phase lattices with
Zou-He boundaries.  advance(n) equals n single steps bit for bit, and with
Zou-He boundaries also the CPU oracle."""
import numpy as np
import pytest

from lbflow_amd import cases as CS
from tests import cases as TC

pytestmark = pytest.mark.gpu


def _engine(spec, solids, dense=False):
    from lbflow_amd.engine import FP64, Engine
    return Engine(CS.lattice(spec), CS.geometry(spec), FP64, solids, dense).init()


def _items(geom, solids):
    """Entries of the two-phase step's work order: the fluid sites, and with
    streamed solids the solid ones, each padded to waves of 64 (one region)."""
    wave = lambda n: (n + 63) // 64 * 64
    fluid = int((geom != 255).sum())
    n = wave(fluid) + (wave(geom.size - fluid) if solids else 0)
    assert n <= 1024
    return n


LIMIT = {2: 768, 3: 512}


@pytest.mark.parametrize('shape,phi,eq,solids,harmonic,several', [
    ((7, 8, 8), 0.7, 'MRT', True, True, True), ((7, 8, 8), 0.7, 'MRT', True, False, True),
    ((6, 8, 8), 0.7, 'SRT', True, True, True), ((8, 8, 8), 0.9, 'MRT', False, True, True),
    ((8, 8, 8), 0.7, 'MRT', True, True, False), ((1, 28, 24), 0.8, 'SRT', True, True, True),
    ((1, 28, 24), 0.8, 'MRT', True, True, True), ((1, 31, 24), 0.8, 'SRT', True, True, False),
    ((1, 30, 28), 0.9, 'MRT', False, True, True)])
def test_colour_limits(shape, phi, eq, solids, harmonic, several):
    rng = np.random.default_rng(sum(shape))
    # both phases fluid and a fixed share of solids, so that the entry count is the shape's own
    n = int(np.prod(shape))
    g = np.full(n, 255, np.uint8)
    fluid = rng.permutation(n)[:int(phi * n)]
    g[fluid] = np.where(rng.random(fluid.size) < 0.5, 75, 76)
    labels = [CS.label_line(75, 'GV', 1e-5, 1, 0), CS.label_line(76, 'VD', phase=1), CS.label_line(255, 'SD', 60)]
    kw = dict(viscosity_interpolation='harmonic', tau=(0.9, 0.6)) if harmonic else dict(tau=(1.0, 1.0))
    spec = CS.make('limit', g.reshape(shape), labels, model='color', eq=eq, sigma=1e-3, beta=0.7, **kw)
    limit = LIMIT[2 if shape[0] == 1 else 3]
    items = _items(g, solids)
    assert (items <= limit) == several and limit - 64 <= items <= limit + 64
    a, b = _engine(spec, solids), _engine(spec, solids)
    for n in (3, 40, 515):
        a.advance(n)
        for _ in range(n):
            b.step(0)
        assert a.t == b.t and a.status()[0] == b.status()[0] == 0
        assert np.array_equal(a.populations().view(np.uint64), b.populations().view(np.uint64))


@pytest.mark.parametrize('spec', TC.zouhe_cases(nx=12, ny=7, nz=6), ids=lambda s: s['name'])
def test_zouhe_advance(spec):
    case, geom = CS.lattice(spec), CS.geometry(spec)
    assert geom.size <= (1024 if case['D'] == 2 else 512)
    from oracle.pyoracle import Oracle
    a, single, orc = _engine(spec, True), _engine(spec, True), Oracle(case, geom).init()
    f, fsingle = _engine(spec, False, True), _engine(spec, False, True)
    for n in (1, 2, 7, 150):
        a.advance(n)
        f.advance(n)
        for _ in range(n):
            single.step(0)
            fsingle.step(0)
        orc.step(n)
        pa, po = a.populations(), orc.populations()
        assert np.array_equal(pa.view(np.uint64), single.populations().view(np.uint64))
        assert np.array_equal(pa.view(np.uint64), po.view(np.uint64))
        assert np.array_equal(f.populations().view(np.uint64), fsingle.populations().view(np.uint64))
    assert a.status()[0] == 0 and f.status()[0] == 0
