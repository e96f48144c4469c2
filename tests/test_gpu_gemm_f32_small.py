"""f32 products of few rows or columns on small tiles with k split inside the workgroup (gemm_f32_small.hip)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["n", "t", "p"])
@pytest.mark.parametrize("m,n,k", [
    (1, 5, 1), (33, 17, 31), (31, 16, 33),        # less than a stage of k; tiles that hang over both ends
    (64, 512, 784), (16, 690, 230), (9, 228, 114),  # rows on 16-byte boundaries and off them
    (64, 1000, 516), (117, 129, 1027),            # more than a stage a wavefront, an uneven last share
    (300, 63, 257), (171, 342, 704), (256, 320, 1280),
])
def test_small_tiles(hip, layout, m, n, k):
    """Every layout at sizes where tiles and stages end raggedly, with and without an offset that takes the operands off 16-byte
    boundaries, against float64: a sum of k products is off by at most k + 1 roundings of the sum of magnitudes."""
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a, b = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(k, n)).astype(np.float32)
    bias, res = rng.normal(size=n).astype(np.float32), rng.normal(size=(m, n)).astype(np.float32)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    plain, bound = a64 @ b64, (k + 1) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    for shift in (0, 1):
        place = lambda v: hip.DeviceBuffer.from_array(np.concatenate([np.zeros(shift, np.float32), np.ascontiguousarray(v).ravel()]))
        d_a, d_b = place(a.T if layout == "t" else a), place(b.T if layout == "p" else b)
        d_bias, d_res = place(bias), place(res)
        out = hip.DeviceBuffer.from_array(np.full(m * n + 64, 7.5, np.float32))
        pa, pb = d_a.at(4 * shift), d_b.at(4 * shift)
        if layout == "t":
            hip.gemm_f32_dev(m, n, k, 0.5, True, pa, pb, out)
            want, slack = 0.5 * plain, 0.5 * bound
        else:
            call = hip.gemm_prepacked_bias_act_f32_dev if layout == "p" else hip.gemm_bias_act_f32_dev
            call(m, n, k, 1, pa, pb, d_bias.at(4 * shift), d_res.at(4 * shift), out)
            pre = plain + bias + res
            want, slack = np.maximum(pre, 0), bound + 2.0 ** -22 * (np.abs(pre) + np.abs(res) + np.abs(bias))
        hip.device_synchronize()
        got = out.to_array(np.float32, m * n + 64)
        assert (got[m * n:] == 7.5).all(), "stores past the result"
        assert (np.abs(got[:m * n].reshape(m, n) - want) <= slack).all(), f"shift {shift}"


@pytest.mark.parametrize("layout", ["n", "t", "p"])
def test_non_finite_values_stay_in_their_rows(hip, layout):
    """k = 33 ends inside a stage and inside a 16-byte piece: what lies behind a row's last value is not multiplied by zero."""
    m, n, k = 40, 35, 33
    rng = np.random.default_rng(2)
    a, b = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(k, n)).astype(np.float32)
    a[8, 0], a[39, 32], b[0, 12] = np.inf, np.nan, -np.inf
    d_a = hip.DeviceBuffer.from_array(np.ascontiguousarray(a.T if layout == "t" else a))
    d_b = hip.DeviceBuffer.from_array(np.ascontiguousarray(b.T if layout == "p" else b))
    out = hip.DeviceBuffer(m * n * 4)
    if layout == "t":
        hip.gemm_f32_dev(m, n, k, 1.0, True, d_a, d_b, out)
    elif layout == "p":
        hip.gemm_prepacked_bias_act_f32_dev(m, n, k, 0, d_a, d_b, None, None, out)
    else:
        hip.gemm_bias_act_f32_dev(m, n, k, 0, d_a, d_b, None, None, out)
    hip.device_synchronize()
    bad = ~np.isfinite(out.to_array(np.float32, m * n).reshape(m, n))
    want = np.zeros((m, n), bool)
    want[8], want[39], want[:, 12] = True, True, True
    assert (bad == want).all()
