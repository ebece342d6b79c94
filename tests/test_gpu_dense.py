"""GPU matvec_q / matmul_q on dense F32, F16 and BF16 rows (ops.rs:87-98,
131-154, 600-623) against the product in float64.  Bar per element: fp32 sums
of n products of exactly widened weights.  From a product to y a term passes
at most 32 roundings at the sizes here: one column, a chain of a wavefront's
steps (512 elements, F32 256: at most 17), 3 adds over the piece, 6 over the
lanes, 4 over up to 8 wavefronts; several, up to 8 products in a chain, 3
adds over the eight chains, a wavefront's steps (128 elements, F32 and more
than 4 columns 64: at most 9), 2 over the lanes, 6 over up to 16
wavefronts.  32 * 2^-24 = 1.9e-6 of sum_i |w_i x_i|: the bar is 2e-6."""
import numpy as np
import pytest

from ouroboros_amd._lib import call
from ouroboros_amd.device import DeviceBuffer
from ouroboros_amd.quant import QuantKind, bf16_bits_to_f32, f32_to_bf16_bits

pytestmark = pytest.mark.gpu


def weights(rng, kind, out_len, in_len):
    w = (rng.standard_normal((out_len, in_len)) / np.sqrt(in_len)).astype(np.float32)
    if kind == QuantKind.F16:
        h = w.astype(np.float16)
        return h.astype(np.float64), h.view(np.uint8).reshape(-1)
    if kind == QuantKind.BF16:
        b = f32_to_bf16_bits(w)
        return bf16_bits_to_f32(b).astype(np.float64), b.view(np.uint8).reshape(-1)
    return w.astype(np.float64), w.view(np.uint8).reshape(-1)


def run(payload, kind, out_len, in_len, x, offset=0):
    k = x.shape[0]
    buf = DeviceBuffer((payload.size + 16,), np.uint8)
    host = np.zeros(payload.size + 16, np.uint8)
    host[offset:offset + payload.size] = payload
    buf.upload(host)
    xd, y = DeviceBuffer.from_host(x), DeviceBuffer((k, out_len), np.float32)
    call("ouro_matmul_q", buf.ptr + offset, int(kind), out_len, in_len, xd.ptr, k, y.ptr, None)
    return y.download().reshape(k, out_len)


# steps (one, whole, a short last one, fewer elements than a step), 16-row tiles
# (one row, a ragged last tile), 1..4 columns and groups of 16 with a ragged last
# one, rows that start at odd elements; one column: 1 and 4 rows a workgroup, of
# several wavefronts and of one (more than 16380 rows)
@pytest.mark.parametrize("kind", [QuantKind.F32, QuantKind.F16, QuantKind.BF16], ids=lambda k: k.name)
@pytest.mark.parametrize("out_len,in_len,k", [(1, 1, 1), (16, 128, 4), (17, 129, 5), (33, 1231, 3), (100, 2560, 16),
                                              (67, 4099, 17), (5003, 640, 1), (70000, 127, 2), (9000, 1030, 1),
                                              (50, 7, 1), (40, 3, 6), (200, 1541, 1), (31, 515, 2),
                                              (16399, 1541, 1)])
@pytest.mark.parametrize("offset", [0, 2])
def test_dense_columns(gpu, kind, out_len, in_len, k, offset):
    rng = np.random.default_rng(out_len + in_len + k)
    w, payload = weights(rng, kind, out_len, in_len)
    x = rng.standard_normal((k, in_len)).astype(np.float32)
    got = run(payload, kind, out_len, in_len, x, 2 * offset if kind == QuantKind.F32 else offset)
    xs = x.astype(np.float64)
    assert (np.abs(got - xs @ w.T) <= 2e-6 * (np.abs(xs) @ np.abs(w).T)).all()


@pytest.mark.parametrize("kind", [QuantKind.F32, QuantKind.F16, QuantKind.BF16], ids=lambda k: k.name)
@pytest.mark.parametrize("k", [1, 3, 6])
def test_dense_non_finite_and_tiny(gpu, kind, k):
    """An infinity or NaN in x reaches its own column only and one in W its
    own row only; products below fp32's normal range and weights below the
    kind's are kept."""
    in_len, out_len = 300, 20

    def stored(w):  # the kind's bytes of w and the values they hold
        if kind == QuantKind.F32:
            return w.astype(np.float64), w.view(np.uint8).reshape(-1)
        bits = w.astype(np.float16).view(np.uint16) if kind == QuantKind.F16 else f32_to_bf16_bits(w)
        vals = bits.view(np.float16) if kind == QuantKind.F16 else bf16_bits_to_f32(bits)
        return vals.astype(np.float64).reshape(w.shape), bits.view(np.uint8).reshape(-1)

    rng = np.random.default_rng(k)
    w = rng.uniform(0.5, 1.0, (out_len, in_len)).astype(np.float32)
    x = rng.uniform(0.5, 1.0, (k, in_len)).astype(np.float32)
    w[3, 7], w[5, 299], x[k - 1, 290] = np.inf, np.nan, -np.inf
    w64, payload = stored(w)
    got = run(payload, kind, out_len, in_len, x)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w64.T
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert np.allclose(got[ok], want[ok], rtol=2e-6, atol=0)  # all terms positive
    # subnormal products: each is a whole number of 2^-149, rounded once
    tiny = np.full((out_len, in_len), 1e-20 if kind != QuantKind.F16 else 2.0 ** -14, np.float32)
    xt = np.full((k, in_len), 1e-20 if kind != QuantKind.F16 else 1e-36, np.float32)
    w64, payload = stored(tiny)
    got = run(payload, kind, out_len, in_len, xt)
    assert np.allclose(got, xt.astype(np.float64) @ w64.T, rtol=1e-3, atol=0)
    # subnormal weights of the kind itself
    low = np.full((out_len, in_len), {QuantKind.F32: 1e-41, QuantKind.F16: 3e-7, QuantKind.BF16: 1e-39}[kind], np.float32)
    xl = rng.uniform(0.5, 1.0, (k, in_len)).astype(np.float32) * np.float32(1e10)
    w64, payload = stored(low)
    assert (w64 != 0).all()
    assert np.allclose(run(payload, kind, out_len, in_len, xl), xl.astype(np.float64) @ w64.T, rtol=2e-6, atol=0)


@pytest.mark.parametrize("kind", [QuantKind.F32, QuantKind.BF16], ids=lambda k: k.name)
@pytest.mark.parametrize("out_len,in_len", [(4096, 2050), (600, 3001), (33, 129)])
def test_dense_column_in_any_number(gpu, kind, out_len, in_len):
    """A column has the same bits among two, three or four columns, and the
    same among any larger number (one column, these and those are summed in
    three orders)."""
    rng = np.random.default_rng(out_len)
    _, payload = weights(rng, kind, out_len, in_len)
    x = rng.standard_normal((40, in_len)).astype(np.float32)
    for few, many in (((2, 3), 4), ((5, 16, 17, 33), 40)):
        whole = run(payload, kind, out_len, in_len, x[:many])
        for k in few:
            assert np.array_equal(run(payload, kind, out_len, in_len, x[:k]), whole[:k]), k
