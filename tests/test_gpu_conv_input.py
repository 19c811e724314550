"""The input layer (8 to 32 channels, BF16 output, sides from 16) equals the
FP32-output direct kernel (pinned against a loop reference in
test_gpu_surrogate.py) rounded to BF16, bit for bit: the smallest side, several
samples, wider rows, and rows that are not whole 16-byte units."""
import numpy as np
import pytest

from lbflow_amd import surrogate as S
from lbflow_amd.engine import Buffer

pytestmark = pytest.mark.gpu


def _bf16(x):
    """float32 -> BF16 bits, nearest even."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


@pytest.mark.parametrize('side,n,in_extra,out_extra,relu', [
    (16, 1, 0, 0, 1), (16, 3, 8, 0, 0), (32, 2, 0, 32, 1), (64, 1, 0, 0, 0), (16, 2, 0, 4, 1), (8, 2, 0, 0, 1)])
def test_input_layer_equals_direct_kernel(side, n, in_extra, out_extra, relu):
    L = S.lib()
    rng = np.random.default_rng(side + n)
    nv = n * side ** 3
    x = Buffer((nv, 8 + in_extra), np.uint16, _bf16(rng.standard_normal((nv, 8 + in_extra), dtype=np.float32)))
    w = np.zeros((32, 224), np.uint16)
    w[:, :216] = _bf16(rng.standard_normal((32, 216), dtype=np.float32) * 0.1)
    dw, b = Buffer(w.shape, np.uint16, w), Buffer((32,), np.float32, rng.standard_normal(32).astype(np.float32))
    got = []
    for f32 in (0, 1):
        out = Buffer((nv, 32 + out_extra), np.float32 if f32 else np.uint16)
        rc = L.lbf_conv3d_forward(8, 32, 27, side, n, x.ptr.value + 2 * in_extra, 8 + in_extra, dw.ptr, b.ptr,
                                  out.ptr, 32 + out_extra, relu, f32)
        assert rc == 0, L.lbf_net_error(None)
        got.append(out.numpy())
    assert np.array_equal(got[0][:, :32], _bf16(got[1][:, :32]))
    assert not got[0][:, 32:].any()   # channels outside the range untouched
