"""3x3x3 convolutions of few voxels at sides from 8: one sample alone (a wave
per 16 x 16 results) equals, bit for bit, the same sample inside a batch that
the tiled kernels take, in both output types.  (Splits over input channels
occur in the networks of test_gpu_surrogate.py.)"""
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
    (32, 32, 8, 65, 0, 0), (64, 32, 8, 24, 64, 0), (384, 128, 8, 8, 0, 0), (256, 256, 8, 5, 0, 32), (32, 64, 16, 3, 0, 0),
    (96, 32, 16, 3, 32, 8)])
@pytest.mark.parametrize('f32', [False, True])
def test_sample_alone_equals_in_batch(cin, cout, side, n, in_extra, out_extra, f32):
    L = S.lib()
    rng = np.random.default_rng(cin + 7 * cout + side + n)
    sv = side ** 3
    x = _bf16(rng.standard_normal((n * sv, cin + in_extra), dtype=np.float32))
    w = Buffer((cout, 27 * cin), np.uint16, _bf16(rng.standard_normal((cout, 27 * cin), dtype=np.float32) * 0.05))
    b = Buffer((cout,), np.float32, rng.standard_normal(cout).astype(np.float32))

    def run(part, samples):
        xin = Buffer(part.shape, np.uint16, part)
        out = Buffer((samples * sv, cout + out_extra), np.float32 if f32 else np.uint16)
        rc = L.lbf_conv3d_forward(cin, cout, 27, side, samples, xin.ptr.value + 2 * in_extra, cin + in_extra, w.ptr,
                                  b.ptr, out.ptr, cout + out_extra, 1, int(f32))
        assert rc == 0, L.lbf_net_error(None)
        return out.numpy()

    whole = run(x, n)
    for s in (0, n - 1):
        alone = run(x[s * sv:(s + 1) * sv], 1)
        assert np.array_equal(alone, whole[s * sv:(s + 1) * sv])
        assert not alone[:, cout:].any()   # channels outside the range untouched
