"""BF16-output 3x3x3 convolutions at sides from 16 (the rows kernel) equal the
FP32-output ones (the halo-tile kernel, pinned against a loop reference in
test_gpu_surrogate.py) rounded to BF16, bit for bit: both add the same
products in the same order.  Sides and samples at which a workgroup's block
wraps around the box, is the whole row, or starts a further sample; wider
rows; and rows whose strides are not whole 16-byte units."""
import numpy as np
import pytest

from lbflow_amd import surrogate as S
from lbflow_amd.engine import Buffer

pytestmark = pytest.mark.gpu


def _bf16(x):
    """float32 -> BF16 bits, nearest even."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


@pytest.mark.parametrize('cin,cout,side,n,in_extra,out_extra', [
    (32, 32, 16, 1, 0, 0), (64, 128, 16, 3, 32, 0), (128, 384, 16, 1, 0, 64), (384, 128, 16, 2, 0, 0),
    (32, 96, 32, 1, 0, 32), (192, 64, 32, 2, 64, 0), (96, 32, 64, 1, 0, 8), (64, 32, 32, 1, 0, 4), (32, 64, 16, 2, 0, 1)])
def test_rows_equal_halo_kernel(cin, cout, side, n, in_extra, out_extra):
    L = S.lib()
    rng = np.random.default_rng(cin + 7 * cout + side + n)
    nv = n * side ** 3
    x = Buffer((nv, cin + in_extra), np.uint16, _bf16(rng.standard_normal((nv, cin + in_extra), dtype=np.float32)))
    w = Buffer((cout, 27 * cin), np.uint16, _bf16(rng.standard_normal((cout, 27 * cin), dtype=np.float32) * 0.05))
    b = Buffer((cout,), np.float32, rng.standard_normal(cout).astype(np.float32))
    got = []
    for f32 in (0, 1):
        out = Buffer((nv, cout + out_extra), np.float32 if f32 else np.uint16)
        rc = L.lbf_conv3d_forward(cin, cout, 27, side, n, x.ptr.value + 2 * in_extra, cin + in_extra, w.ptr, b.ptr,
                                  out.ptr, cout + out_extra, 1, f32)
        assert rc == 0, L.lbf_net_error(None)
        got.append(out.numpy())
    assert np.array_equal(got[0][:, :cout], _bf16(got[1][:, :cout]))
    assert not got[0][:, cout:].any()   # channels outside the range untouched
