"""Lattices whose FP64 steps run several to a launch: advance(n) equals n single
steps bit for bit in both models, for sizes up to and
beyond the limit, rows of one site, no solid and hardly any fluid, an odd and
an even number of steps and more than one launch; and a failure is recorded at
the step at which single steps record it."""
import numpy as np
import pytest

from lbflow_amd import cases as CS

pytestmark = pytest.mark.gpu


def _spec(shape, phi, eq):
    rng = np.random.default_rng(sum(shape))
    g = np.where(rng.random(shape) < phi, np.where(rng.random(shape) < 0.5, 75, 76), 255).astype(np.uint8)
    labels = [CS.label_line(75, 'GV', 1e-5, 1, 0), CS.label_line(76, 'VD'), CS.label_line(255, 'SD', 60)]
    return CS.make('small', g, labels, model='scsp', eq=eq, tau=(0.8,))


def _engine(spec, solids):
    from lbflow_amd.engine import FP64, Engine
    return Engine(CS.lattice(spec), CS.geometry(spec), FP64, solids).init()


def _colour(shape, phi, eq, harmonic):
    rng = np.random.default_rng(sum(shape))
    g = np.where(rng.random(shape) < phi, np.where(rng.random(shape) < 0.5, 75, 76), 255).astype(np.uint8)
    labels = [CS.label_line(75, 'GV', 1e-5, 1, 0), CS.label_line(76, 'VD', phase=1), CS.label_line(255, 'SD', 60)]
    kw = dict(viscosity_interpolation='harmonic', tau=(0.9, 0.6)) if harmonic else dict(tau=(1.0, 1.0))
    return CS.make('small', g, labels, model='color', eq=eq, sigma=1e-3, beta=0.7, **kw)


@pytest.mark.parametrize('shape,phi,eq,solids,harmonic', [
    ((1, 9, 7), 0.6, 'MRT', True, False), ((1, 24, 32), 1.0, 'MRT', True, True), ((1, 31, 24), 0.8, 'SRT', True, True),
    ((1, 32, 32), 0.6, 'MRT', False, False), ((8, 8, 8), 0.7, 'MRT', True, True), ((8, 8, 8), 1.0, 'SRT', False, False),
    ((8, 8, 9), 0.4, 'MRT', False, False), ((4, 4, 4), 0.0, 'MRT', True, False)])
def test_colour_advance_equals_single_steps(shape, phi, eq, solids, harmonic):
    spec = _colour(shape, phi, eq, harmonic)
    a, b = _engine(spec, solids), _engine(spec, solids)
    for n in (1, 2, 7, 40):
        a.advance(n)
        for _ in range(n):
            b.step(0)
        assert a.t == b.t and a.status()[0] == b.status()[0]
        assert np.array_equal(a.populations().view(np.uint64), b.populations().view(np.uint64))


@pytest.mark.parametrize('shape,phi,eq,solids', [
    ((1, 1, 1), 1.0, 'MRT', True), ((1, 7, 9), 0.6, 'MRT', True), ((1, 16, 32), 1.0, 'SRT', True),
    ((1, 19, 27), 0.8, 'MRT', True), ((1, 32, 32), 0.9, 'MRT', True),
    ((1, 41, 25), 0.8, 'SRT', True), ((8, 8, 8), 0.7, 'MRT', True), ((8, 8, 8), 1.0, 'SRT', False),
    ((5, 13, 1), 0.5, 'MRT', False), ((4, 5, 3), 0.03, 'MRT', False)])
def test_advance_equals_single_steps(shape, phi, eq, solids):
    spec = _spec(shape, phi, eq)
    a, b = _engine(spec, solids), _engine(spec, solids)
    for n in (1, 2, 7, 516):
        a.advance(n)
        for _ in range(n):
            b.step(0)
        assert a.t == b.t
        assert np.array_equal(a.populations().view(np.uint64), b.populations().view(np.uint64))


def test_failure_step():
    spec = _spec((1, 9, 9), 1.0, 'MRT')
    first = []
    for single in (False, True):
        e = _engine(spec, True)
        p = e.populations()
        p[40] = 1.7e308
        e.set_populations(p, 5)
        if single:
            for _ in range(6):
                e.step(0)
        else:
            e.advance(6)
        bits, f = e.status()
        first.append((bits, [int(x) for x in f]))
    assert first[0][0] and first[0] == first[1]
