"""FP64 steps several to a launch, where their rules end: two-phase work orders
whose padded entries just fill or just miss the limit (the count is asserted,
so that each case runs the kernel it is there for), per-site relaxation times
in D3Q19, more steps than one launch holds.  advance(n) equals n single steps bit
for bit."""
import numpy as np
import pytest

from lbflow_amd import cases as CS

pytestmark = pytest.mark.gpu


def _engine(spec, solids):
    from lbflow_amd.engine import FP64, Engine
    return Engine(CS.lattice(spec), CS.geometry(spec), FP64, solids).init()


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
