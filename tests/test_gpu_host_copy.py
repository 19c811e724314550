"""Large results arrive whole in ordinary host memory: fields around the size at
which the copy is split over threads and past whole chunks, several engines
copying at once, a handle outliving the others, and the network's parameters
in the caller's layout."""
import threading

import numpy as np
import pytest

from lbflow_amd import cases as CS
from lbflow_amd import surrogate as S
from lbflow_amd.engine import FP32, Engine

pytestmark = pytest.mark.gpu


def _engine(ny, nx):
    """D2Q9 at t = 0, where a site's velocity depends on its label alone (the
    rounding of half its force): the value of each label comes from a lattice
    of three sites, one per label, too small for the threads."""
    rng = np.random.default_rng(ny)
    g = rng.choice(np.array([10, 11, 12], np.uint8), size=(ny, nx))
    force = {10: 1e-5, 11: 3e-5, 12: 7e-5}
    spec = CS.make('copy', g, [CS.label_line(k, 'GV', f, 1, 0) for k, f in force.items()], tau=(0.8,))
    keys = np.array(list(force), np.uint8).reshape(1, 3)
    one = CS.make('labels', keys, spec['indices'], tau=(0.8,))
    want = np.zeros(256)
    want[keys.ravel()] = Engine(CS.lattice(one), keys.ravel(), FP32, False).init().fields()[2][1]
    assert len(set(want[keys.ravel()])) == 3
    return Engine(CS.lattice(spec), g.ravel(), FP32, False).init(), want[g.ravel()]


def _check(eng, want):
    rho, _, u = eng.fields()
    assert np.array_equal(u[1], want) and not u[0].any()
    assert np.all(rho == 1.0)


@pytest.mark.parametrize('ny,nx', [(1, 16), (524, 1000), (1024, 512), (1024, 1025), (1500, 1501)])
def test_fields_whole(ny, nx):
    eng, want = _engine(ny, nx)
    _check(eng, want)


def test_several_engines_at_once():
    pairs = [_engine(1100 + 7 * k, 1201) for k in range(3)]
    failed = []

    def run(p):
        try:
            for _ in range(3):
                _check(*p)
        except AssertionError as e:   # pragma: no cover
            failed.append(e)
    threads = [threading.Thread(target=run, args=(p,)) for p in pairs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    for eng, _ in pairs[:2]:
        eng.close()
    _check(*pairs[2])


def test_parameters_in_the_callers_layout():
    net = S.Net(side=8, capacity=1, seed=3)
    p = np.random.default_rng(5).standard_normal(net.n_params).astype(np.float32)
    net.set_params(p)
    assert np.array_equal(net.params(), p)
