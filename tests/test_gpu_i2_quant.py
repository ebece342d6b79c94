"""Quantisation of activations ahead of a ternary product: whole-integer and
bit-exact results, whichever kernel runs.  The row kernel with 4-element loads
(rows of whole groups, 256 to 8192) at its register-count edges, the element
loop on either side and on odd lengths or addresses; and a resident weight's matvec,
which rounds x inside the product below a size, against the two calls
ouro_act_quant_i8 and ouro_gemm_i2 at every row length that a weight takes."""
import numpy as np
import pytest

from ouroboros_amd import _lib, ops
from ouroboros_amd._lib import DT_BF16, DT_F32, call
from ouroboros_amd.device import DeviceBuffer
from ouroboros_amd.quant import QuantKind, bf16_bits_to_f32, f32_to_bf16_bits, i2_pack

pytestmark = pytest.mark.gpu


def inputs(rng, rows, n):
    x = rng.standard_normal((rows, n)).astype(np.float32)
    x[rng.random((rows, n)) < 0.01] *= 20.0
    x[0] = 0.0  # the smallest scale
    return x


@pytest.mark.parametrize("n", [1, 4, 7, 252, 256, 1020, 1024, 2048, 2052, 4096, 4100, 6912, 8192, 8196, 4098])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("off", [0, 1])  # bytes that xq lies past its boundary
@pytest.mark.parametrize("x_off", [0, 1, 2])  # elements that x lies past a 16-byte boundary
def test_act_quant_rows(gpu, orc, n, bf16, off, x_off):
    rows = 5
    x = inputs(np.random.default_rng(n), rows, n)
    bits = f32_to_bf16_bits(x)
    if bf16:
        x = bf16_bits_to_f32(bits).reshape(rows, n)
    want_q, want_s = orc.act_quant_i8(x)
    src = (bits if bf16 else x).reshape(-1)
    xd = DeviceBuffer.from_host(np.concatenate([np.zeros(x_off, src.dtype), src]))
    xp = xd.ptr + x_off * src.itemsize
    q, s = DeviceBuffer((rows * n + 16,), np.int8), DeviceBuffer((rows,), np.float32)
    call("ouro_act_quant_i8", xp, DT_BF16 if bf16 else DT_F32, rows, n, q.ptr + off, s.ptr, None)
    assert np.array_equal(q.download()[off:off + rows * n].reshape(rows, n), want_q)
    assert np.array_equal(s.download().view(np.uint32), want_s.view(np.uint32))


@pytest.mark.parametrize("out_len,in_len", [(1, 256), (9, 512), (33, 1024), (70, 2048), (64, 2560), (65, 3072), (40, 4096),
                                            (31, 5120), (17, 6144), (100, 6912), (8, 8192), (61440, 1024), (61448, 1024),
                                            (98304, 256), (98305, 256), (8192, 5120), (8193, 5120), (9000, 8192)])
def test_matvec_rounds_x_itself(gpu, out_len, in_len):
    """Every row length that a weight takes, and both sides of the size rule:
    61440 tiles of 8 rows times 256-element groups and four, 1024 tiles from
    17 groups on."""
    rng = np.random.default_rng(out_len + in_len)
    w = rng.integers(-1, 2, size=(out_len, in_len)).astype(np.int8)
    h = ops.Weight(QuantKind.I2, i2_pack(w), out_len, in_len, w_scale=0.7)
    x = inputs(rng, 2, in_len)
    x[1, in_len - 1] = 1e30  # every other element rounds to zero
    # the handle's payload: tiled codes, then the scale
    payload = _lib.lib().ouro_weight_payload(h.handle)
    scale = payload + _lib.lib().ouro_i2_tiled_bytes(out_len, in_len)
    rows = np.concatenate([x, inputs(rng, 2, in_len)[1:]])
    for x_off, row in enumerate(rows):  # the product reads x at any 4-byte boundary
        xd = DeviceBuffer.from_host(np.concatenate([np.zeros(x_off, np.float32), row]))
        xp = xd.ptr + 4 * x_off
        q, s = DeviceBuffer((in_len,), np.int8), DeviceBuffer((1,), np.float32)
        y, y2 = DeviceBuffer((out_len,), np.float32), DeviceBuffer((out_len,), np.float32)
        call("ouro_weight_matvec", h.handle, xp, y.ptr, None)
        call("ouro_act_quant_i8", xp, DT_F32, 1, in_len, q.ptr, s.ptr, None)
        call("ouro_gemm_i2", payload, out_len, in_len, scale, q.ptr, s.ptr, 1, y2.ptr, None, None)
        assert np.array_equal(y.download().view(np.uint32), y2.download().view(np.uint32))


@pytest.mark.parametrize("out_len,in_len", [(2560, 2560), (8192, 8192), (1000, 4096), (6000, 1024)])
@pytest.mark.parametrize("shift", [0, 40, -40])
def test_matvec_in_place(gpu, out_len, in_len, shift):
    """y over x, whole or in part, by a handle, a payload and without allocation: the bits of y elsewhere."""
    rng = np.random.default_rng(out_len)
    w = rng.integers(-1, 2, size=(out_len, in_len)).astype(np.int8)
    h = ops.Weight(QuantKind.I2, i2_pack(w), out_len, in_len, w_scale=0.7)
    payload = _lib.lib().ouro_weight_payload(h.handle)
    x = inputs(rng, 2, in_len)[1]
    xd, y = DeviceBuffer.from_host(x), DeviceBuffer((out_len,), np.float32)
    call("ouro_weight_matvec", h.handle, xd.ptr, y.ptr, None)
    want = y.download()
    at, n = 64, 128 + max(out_len, in_len)
    host = np.zeros(n, np.float32)
    host[at:at + in_len] = x
    buf = DeviceBuffer((n,), np.float32)
    xp, yp = buf.ptr + 4 * at, buf.ptr + 4 * (at + shift)
    for fn, *a in (("ouro_weight_matvec", h.handle), ("ouro_matvec_q", payload, int(QuantKind.I2), out_len, in_len),
                   ("ouro_matvec_q_noalloc", payload, int(QuantKind.I2), out_len, in_len)):
        buf.upload(host)
        call(fn, *a, xp, yp, None)
        got = buf.download()[at + shift:at + shift + out_len]
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), fn
