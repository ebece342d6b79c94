"""GPU matvec_q / matmul_q on dense F32, F16 and BF16 rows (ops.rs:87-98,
131-154, 600-623) against the product in float64.  Bar per element: fp32
sums of n products of exactly widened weights differ from the exact sum by
at most a few roundings of sum_i |w_i x_i| (chains of 32 products a step, 4
sums a step, then at most in_len / 128 steps over 16 wavefronts); 2e-6 of
that sum covers the longest rows here many times over."""
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


# steps of 128 elements (one, whole, a short last one, fewer elements than a
# step), 16-row tiles (one row, a ragged last tile), 1..4 columns and groups
# of 16 with a ragged last one, rows that start at odd elements
@pytest.mark.parametrize("kind", [QuantKind.F32, QuantKind.F16, QuantKind.BF16], ids=lambda k: k.name)
@pytest.mark.parametrize("out_len,in_len,k", [(1, 1, 1), (16, 128, 4), (17, 129, 5), (33, 1231, 3), (100, 2560, 16),
                                              (67, 4099, 17), (5003, 640, 1), (70000, 127, 2), (9000, 1030, 1),
                                              (50, 7, 1), (40, 3, 6), (200, 1541, 1), (31, 515, 2)])
@pytest.mark.parametrize("offset", [0, 2])
def test_dense_columns(gpu, kind, out_len, in_len, k, offset):
    rng = np.random.default_rng(out_len + in_len + k)
    w, payload = weights(rng, kind, out_len, in_len)
    x = rng.standard_normal((k, in_len)).astype(np.float32)
    got = run(payload, kind, out_len, in_len, x, 2 * offset if kind == QuantKind.F32 else offset)
    xs = x.astype(np.float64)
    assert (np.abs(got - xs @ w.T) <= 2e-6 * (np.abs(xs) @ np.abs(w).T)).all()


@pytest.mark.parametrize("k", [1, 6])
def test_dense_non_finite_and_tiny(gpu, k):
    """An infinity or NaN in x reaches its own column only and one in W its
    own row only; products below fp32's normal range are kept."""
    in_len, out_len = 300, 20
    rng = np.random.default_rng(k)
    w = rng.uniform(0.5, 1.0, (out_len, in_len)).astype(np.float32)
    x = rng.uniform(0.5, 1.0, (k, in_len)).astype(np.float32)
    w[3, 7], w[5, 299], x[k - 1, 290] = np.inf, np.nan, -np.inf
    got = run(w.view(np.uint8).reshape(-1), QuantKind.F32, out_len, in_len, x)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.T.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    tiny = np.full((out_len, in_len), 1e-20, np.float32)
    got = run(tiny.view(np.uint8).reshape(-1), QuantKind.F32, out_len, in_len, np.full((k, in_len), 1e-20, np.float32))
    assert np.allclose(got, in_len * 1e-40, rtol=1e-3, atol=0)


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
