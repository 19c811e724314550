"""FP64 colour steps at the edges of their work order: lattices whose fluid and
solid sites just fill, or just miss, waves of 64, workgroups and regions, with
no fluid or no solid at all, and with and without streamed solids, bit for bit
against the CPU oracle (the operators, the paired recolouring divisions and
the wave order must not change a bit)."""
import numpy as np
import pytest

from lbflow_amd import cases as CS

pytestmark = pytest.mark.gpu


def _case(nz, ny, nx, phi, eq, tau, seed, harmonic=False):
    rng = np.random.default_rng(seed)
    g = np.where(rng.random((nz, ny, nx)) < phi, np.where(rng.random((nz, ny, nx)) < 0.5, 75, 76), 255)
    kw = dict(viscosity_interpolation='harmonic') if harmonic else {}
    return CS.make('order', g.astype(np.uint8),
                   [CS.label_line(75, 'GV', 1e-5, 1, 0), CS.label_line(76, 'VD', phase=1),
                    CS.label_line(255, 'SD', 60)], model='color', eq=eq, tau=tau, sigma=1e-3, beta=0.7, **kw)


@pytest.mark.parametrize('nz,ny,nx,phi,eq,tau,solids', [
    (1, 8, 8, 1.0, 'MRT', (1.0, 1.0), True), (1, 9, 7, 0.5, 'MRT', (0.9, 0.6), True),
    (4, 4, 4, 1.0, 'MRT', (1.0, 1.0), True), (5, 13, 1, 0.6, 'SRT', (0.8, 1.1), True),
    (4, 16, 16, 0.3, 'MRT', (1.0, 1.0), True), (5, 16, 13, 0.9, 'MRT', (1.0, 0.7), True),
    (4, 16, 16, 0.0, 'MRT', (1.0, 1.0), True), (9, 11, 12, 0.25, 'MRT', (1.0, 1.0), False)])
def test_work_order_edges(nz, ny, nx, phi, eq, tau, solids):
    from lbflow_amd.engine import FP64, Engine
    from oracle.pyoracle import Oracle
    spec = _case(nz, ny, nx, phi, eq, tau, 11, harmonic=tau[0] != tau[1])
    case, geom = CS.lattice(spec), CS.geometry(spec)
    eng = Engine(case, geom, FP64, solids).init()
    eng.advance(12)
    orc = Oracle(case, geom).init().step(12)
    a, b = eng.populations(), orc.populations()
    if not solids:   # solid sites are not streamed without LBF_STREAM_SOLIDS
        keep = np.tile(geom != 255, a.size // geom.size)
        a, b = a[keep], b[keep]
    assert np.array_equal(a, b)
