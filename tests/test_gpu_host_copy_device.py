"""Fields and populations copied to device memory instead of the host's arrive
whole, below and above the size from which large host results go through
threads."""
import numpy as np
import pytest

from lbflow_amd import cases as CS
from lbflow_amd.engine import FP64, STEP_FIELDS, Buffer, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape', [(1, 64, 64), (1, 1100, 1003)])
def test_device_destination(shape):
    rng = np.random.default_rng(shape[1])
    g = np.where(rng.random(shape) < 0.9, 75, 255).astype(np.uint8)
    spec = CS.make('dst', g, [CS.label_line(75, 'GV', 1e-5, 1, 0), CS.label_line(255, 'SD', 90)], tau=(0.8,))
    e = Engine(CS.lattice(spec), g.ravel(), FP64, True).init()
    e.step(0).step(STEP_FIELDS)
    rho, _, u = e.fields()
    d_rho, d_u = Buffer((e.N,), np.float64), Buffer(u.shape, np.float64)
    d_pop = Buffer((e.Q * e.N,), np.float64)
    e._check(e.L.lbf_fields(e.h, d_rho.ptr, None, d_u.ptr))
    e._check(e.L.lbf_get_populations(e.h, d_pop.ptr))
    assert np.array_equal(d_rho.numpy(), rho) and np.array_equal(d_u.numpy(), u)
    assert np.array_equal(d_pop.numpy(), e.populations())
