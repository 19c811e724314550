"""3x3x3 forward convolutions split over input channels, and with the ReLU
gradient's gate, at the sizes where the networks run them: through the
library's own launcher, since lbf_conv3d_forward offers neither a workspace
nor a gate.  FP32 results against a float64 product under the bound of FP32
sums; BF16 results, whose kernels may be others, must be those rounded, bit for
bit (the same products in the same order); the workspace is written just as
far as the expected number of splits."""
import ctypes as C

import numpy as np
import pytest

from lbflow_amd import surrogate as S
from lbflow_amd.engine import Buffer

pytestmark = pytest.mark.gpu

ACT_NONE, ACT_GATE = 0, 2


class ConvGeom(C.Structure):   # csrc/conv_types.h
    _fields_ = [('log_s', C.c_uint32), ('nvox', C.c_uint32), ('in_stride', C.c_uint32), ('out_stride', C.c_uint32),
                ('gate', C.c_void_p), ('gate_stride', C.c_uint32), ('kpart', C.c_void_p), ('kpart_floats', C.c_uint32),
                ('out_channels', C.c_uint32)]


def _launcher():
    # lbf::launch_conv_forward(int, int, int, const ConvGeom&, const __bf16*, const __bf16*, const float*, void*, int,
    # bool, hipStream_t)
    fn = getattr(S.lib(), '_ZN3lbf19launch_conv_forwardEiiiRKNS_8ConvGeomEPKDF16bS4_PKfPvibP12ihipStream_t')
    fn.argtypes = [C.c_int] * 3 + [C.c_void_p] * 5 + [C.c_int, C.c_bool, C.c_void_p]
    fn.restype = C.c_int
    return fn


def _bits(x):
    """float32 -> BF16 bits, nearest even."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def _value(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32)


def _products(x, w, side):
    """Periodic 3x3x3 convolution in float64, x [voxel][cin], w [cout][27][cin]."""
    n = x.shape[0] // side ** 3
    v = x.astype(np.float64).reshape(n, side, side, side, -1)
    out = np.zeros((x.shape[0], w.shape[0]))
    for t in range(27):
        moved = np.roll(v, shift=(1 - t // 9, 1 - t // 3 % 3, 1 - t % 3), axis=(1, 2, 3))
        out += moved.reshape(x.shape) @ w[:, t, :].astype(np.float64).T
    return out


class Case:
    def __init__(self, cin, cout, side, n, in_extra, workspace):
        rng = np.random.default_rng(cin + 7 * cout + side + n)
        self.cin, self.cout, self.side, self.nv, self.in_extra = cin, cout, side, n * side ** 3, in_extra
        self.xb = _bits(rng.standard_normal((self.nv, cin + in_extra), dtype=np.float32))
        self.wb = _bits(rng.standard_normal((cout, 27, cin), dtype=np.float32) / np.sqrt(np.float32(27 * cin)))
        self.bias = rng.standard_normal(cout).astype(np.float32)
        self.dx, self.dw = Buffer(self.xb.shape, np.uint16, self.xb), Buffer(self.wb.shape, np.uint16, self.wb)
        self.rng, self.workspace = rng, workspace

    def run(self, act, f32, bias, out_extra=0, gate=None, gate_stride=0):
        out = Buffer((self.nv, self.cout + out_extra), np.float32 if f32 else np.uint16)
        part = None
        if self.workspace:
            part = Buffer((self.workspace,), np.float32, np.full(self.workspace, np.nan, np.float32))
        b = None if bias is None else Buffer(bias.shape, np.float32, bias)
        g = ConvGeom(self.side.bit_length() - 1, self.nv, self.cin + self.in_extra, self.cout + out_extra,
                     gate, gate_stride, part.ptr.value if part else None, self.workspace, 0)
        rc = _launcher()(self.cin, self.cout, 27, C.byref(g), self.dx.ptr.value + 2 * self.in_extra, self.dw.ptr,
                         b.ptr if b else None, out.ptr, act, bool(f32), None)
        assert rc == 0
        r = out.numpy()   # (waits: a blocking copy on the same stream)
        assert not r[:, self.cout:].any()   # channels outside the range untouched
        splits = 1
        if part is not None:
            written = int((~np.isnan(part.numpy())).sum())
            assert written % (self.nv * self.cout) == 0
            splits = max(1, written // (self.nv * self.cout))
        return r[:, :self.cout], splits


# cin, cout, side, samples, expected splits.  BF16 kernels: rows (16-row and
# 32-row blocks), few voxels, halo tiles; FP32: few voxels or halo tiles.
SPLIT = [(192, 64, 16, 2, 2), (384, 128, 16, 1, 4), (64, 64, 32, 1, 2), (256, 128, 16, 1, 8), (64, 32, 16, 10, 2),
         (64, 32, 8, 1, 2), (384, 128, 8, 1, 4), (256, 256, 8, 2, 8), (384, 128, 8, 3, 4)]


@pytest.mark.parametrize('cin,cout,side,n,splits', SPLIT)
def test_splits(cin, cout, side, n, splits):
    c = Case(cin, cout, side, n, 32, 1 << 23)
    want32, s32 = c.run(ACT_NONE, True, c.bias, out_extra=4)
    got16, s16 = c.run(ACT_NONE, False, c.bias, out_extra=8)
    assert (s32, s16) == (splits, splits)
    x, w = _value(c.xb)[:, 32:], _value(c.wb)
    exact = _products(x, w, side) + c.bias
    bound = 27 * cin * 2.0 ** -24 * (_products(np.abs(x), np.abs(w), side) + np.abs(c.bias))
    assert (np.abs(want32 - exact) <= bound).all()
    assert np.array_equal(got16, _bits(want32))


# the same with a gate, and unsplit (no workspace) where the gate rides in the
# rows kernel's own stores: 16-row and 32-row blocks
@pytest.mark.parametrize('cin,cout,side,n,workspace,gate_extra', [
    (192, 64, 16, 2, 0, 0), (64, 64, 32, 1, 0, 32), (128, 384, 16, 1, 0, 8), (32, 96, 32, 1, 0, 0), (32, 32, 16, 20, 0, 64),
    (192, 64, 16, 2, 1 << 23, 32), (64, 64, 32, 1, 1 << 23, 0), (64, 32, 8, 1, 1 << 23, 0), (32, 32, 16, 2, 0, 3),
    (256, 128, 8, 4, 1 << 23, 8), (256, 256, 4, 70, 0, 5)])
def test_gate(cin, cout, side, n, workspace, gate_extra):
    c = Case(cin, cout, side, n, 0, workspace)
    plain, _ = c.run(ACT_NONE, True, np.zeros(cout, np.float32))
    x, w = _value(c.xb), _value(c.wb)
    bound = 27 * cin * 2.0 ** -24 * _products(np.abs(x), np.abs(w), side)
    assert (np.abs(plain - _products(x, w, side)) <= bound).all()
    gb = _bits(c.rng.standard_normal((c.nv, cout + gate_extra), dtype=np.float32))
    gb[c.rng.random(gb.shape) < 0.1] = 0
    gb[c.rng.random(gb.shape) < 0.1] = 0x8000   # -0
    gate = Buffer(gb.shape, np.uint16, gb)
    got, _ = c.run(ACT_GATE, False, None, out_extra=8, gate=gate.ptr.value + 2 * gate_extra, gate_stride=cout + gate_extra)
    assert np.array_equal(got, np.where(_value(gb)[:, gate_extra:] > 0, _bits(plain), 0))
