"""3x3x3 convolutions at sides below 8 against the float64 loop reference:
voxel counts that end inside a 16-voxel tile or a wave's four tiles, on both
sides of the rule between them, and wider rows."""
import numpy as np
import pytest

from lbflow_amd import surrogate as S
from lbflow_amd.engine import Buffer
from oracle import surrogate_ref as R

pytestmark = pytest.mark.gpu


def _bf16(x):
    """float32 -> BF16 bits, nearest even."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def _f64(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


@pytest.mark.parametrize('cin,cout,side,n,in_extra,out_extra', [
    (32, 32, 1, 1, 0, 0), (64, 32, 1, 17, 8, 0), (256, 256, 2, 3, 0, 0), (32, 64, 2, 65, 0, 3), (128, 256, 4, 1, 64, 0),
    (384, 128, 4, 8, 0, 32), (96, 32, 4, 9, 0, 0)])
def test_coarse_sides(cin, cout, side, n, in_extra, out_extra):
    L = S.lib()
    rng = np.random.default_rng(cin + 7 * cout + side + n)
    nv = n * side ** 3
    x = _bf16(rng.standard_normal((nv, cin + in_extra), dtype=np.float32))
    w = _bf16(rng.standard_normal((cout, 27, cin), dtype=np.float32) / np.sqrt(np.float32(27 * cin)))
    b = rng.standard_normal(cout).astype(np.float32)
    dx, dw, db = Buffer(x.shape, np.uint16, x), Buffer((cout, 27 * cin), np.uint16, w), Buffer((cout,), np.float32, b)
    xs = _f64(x)[:, in_extra:].reshape(n, side, side, side, cin)
    want = R.conv_bruteforce(xs, _f64(w), b).reshape(nv, cout)
    # FP32 sums of 27 Cin products: their rounding is at most 27 Cin eps times
    # the sum of the products' sizes
    bound = 27 * cin * 2.0 ** -24 * (R.conv_bruteforce(np.abs(xs), np.abs(_f64(w)), np.abs(b)).reshape(nv, cout))
    got = []
    for f32 in (0, 1):
        out = Buffer((nv, cout + out_extra), np.float32 if f32 else np.uint16)
        rc = L.lbf_conv3d_forward(cin, cout, 27, side, n, dx.ptr.value + 2 * in_extra, cin + in_extra, dw.ptr, db.ptr,
                                  out.ptr, cout + out_extra, 0, f32)
        assert rc == 0, L.lbf_net_error(None)
        got.append(out.numpy())
    assert (np.abs(got[1][:, :cout] - want) <= bound).all()
    assert np.array_equal(got[0][:, :cout], _bf16(got[1][:, :cout]))
    assert not got[0][:, cout:].any()   # channels outside the range untouched
