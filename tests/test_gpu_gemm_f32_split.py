"""f32 products that run on the bf16 matrix cores as sums of three exact bf16 pieces, against float64."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# Rows and columns one off the tile heights (64, 96, 128, 160, 256) and widths (64, 128), terms that are no multiple of 16,
# of 32 (the step pairs) or of 4 (unaligned rows), with and without a split of k over workgroups.
SHAPES = [(1233, 1000, 700), (1021, 1111, 333), (300, 700, 2100), (1576, 768, 3072), (1601, 2050, 515), (2049, 2561, 97),
          (1537, 1535, 769), (65, 4097, 1001), (4097, 33, 1003), (2303, 1388, 1040), (3841, 3970, 290)]


def run(hip, m, n, k, layout, a, b, bias=None, residual=None, activation=0):
    """a (m, k) and b (k, n); layout "n": both as they are, "t": A handed over as its transpose, "p": B as its transpose."""
    d_a = hip.DeviceBuffer.from_array(a.T if layout == "t" else a)
    d_b = hip.DeviceBuffer.from_array(b.T if layout == "p" else b)
    d_bias = None if bias is None else hip.DeviceBuffer.from_array(bias)
    d_res = None if residual is None else hip.DeviceBuffer.from_array(residual)
    d_c = hip.DeviceBuffer.from_array(np.full(m * n + 64, 7.5, np.float32))
    if layout == "t":
        hip.gemm_f32_dev(m, n, k, 1.0, True, d_a, d_b, d_c)
    elif layout == "p":
        hip.gemm_prepacked_bias_act_f32_dev(m, n, k, activation, d_a, d_b, d_bias, d_res, d_c)
    else:
        hip.gemm_bias_act_f32_dev(m, n, k, activation, d_a, d_b, d_bias, d_res, d_c)
    hip.device_synchronize()
    out = d_c.to_array(np.float32, m * n + 64)
    assert (out[m * n:] == 7.5).all(), "wrote past the end of the result"
    return out[:m * n].reshape(m, n)


@pytest.mark.parametrize("layout", ["n", "t", "p"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_against_float64(hip, m, n, k, layout):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(k, n)).astype(np.float32)
    bias = residual = None
    activation = 0
    if layout != "t":
        bias, residual, activation = rng.normal(size=n).astype(np.float32), rng.normal(size=(m, n)).astype(np.float32), 1
    got = run(hip, m, n, k, layout, a, b, bias, residual, activation)
    product = a.astype(np.float64) @ b.astype(np.float64)
    want = product if bias is None else np.maximum(product + bias + residual, 0.0)
    # The sum takes one rounding (at most 2^-24 of itself) per sixteen terms and a few at the end, independent of each
    # other: they add in quadrature.  Leaving out any one of the pieces costs 2^-18 of a product and fails this.
    bound = 2.0 ** -24 * np.sqrt(k / 16 + 8) * np.sqrt(np.mean(product ** 2))
    assert np.sqrt(np.mean((got - want) ** 2)) <= bound
    assert np.abs(got - want).max() <= 8 * bound  # eight standard deviations


@pytest.mark.parametrize("layout", ["n", "t", "p"])
@pytest.mark.parametrize("m,n,k", [(1233, 1000, 700), (300, 700, 2100)])
def test_finite_operands_whose_products_overflow(hip, m, n, k, layout):
    """Every product of 1e25 and more leaves f32: an infinity of its sign, as f32 sums give, which a fused ReLU keeps."""
    rng = np.random.default_rng(8)
    a, b = (rng.uniform(1e25, 2e25, shape).astype(np.float32) for shape in ((m, k), (k, n)))
    b[:, ::3] *= -1.0
    negative = np.broadcast_to(np.arange(n) % 3 == 0, (m, n))
    assert (run(hip, m, n, k, layout, a, b) == np.where(negative, -np.inf, np.inf)).all()
    if layout != "t":
        bias = np.zeros(n, np.float32)
        assert (run(hip, m, n, k, layout, a, b, bias, None, 1) == np.where(negative, 0.0, np.inf)).all()
    # products that just fit, sums that do not, and sums that do
    a[:] = np.float32(2.0 ** 64)
    b[:] = np.float32(2.0 ** 63) * np.where(np.arange(n) % 3 == 0, -1, 1)
    assert (run(hip, m, n, k, layout, a, b) == np.where(negative, -np.inf, np.inf)).all()
    b *= np.float32(2.0 ** -12)
    assert (run(hip, m, n, k, layout, a, b) == np.where(negative, -1.0, 1.0) * k * 2.0 ** 115).all()


@pytest.mark.parametrize("layout", ["n", "t", "p"])
@pytest.mark.parametrize("m,n,k", [(1233, 1000, 700), (300, 700, 2100)])
def test_small_values_beside_ordinary_ones(hip, m, n, k, layout):
    """A value of 1e-36, or a subnormal one, keeps all its bits in a row of ordinary values: the sums below hang on it."""
    rng = np.random.default_rng(12)
    a, b = rng.normal(size=(m, k)).astype(np.float32), np.zeros((k, n), np.float32)
    a[:, 5] = (rng.normal(size=m) * 1e-36).astype(np.float32)
    a[:, k - 2] = (rng.normal(size=m) * 1e-38).astype(np.float32)  # subnormal ones among them
    b[5, ::2] = np.float32(1e20)
    b[k - 2, 1::2] = np.float32(-1.3e20)
    got = run(hip, m, n, k, layout, a, b)
    want = a.astype(np.float64) @ b.astype(np.float64)
    # one product each: rounded once at the end (2^-24), piece products of 2^-24 left out, five roundings of sums 2^-8 its size
    assert (np.abs(got - want) <= 2.02 * 2.0 ** -24 * np.abs(want)).all()
    b[7] = rng.normal(size=n)
    a[:, 7] = (rng.normal(size=m) * 1e-16).astype(np.float32)
    got, want = run(hip, m, n, k, layout, a, b), a.astype(np.float64) @ b.astype(np.float64)
    magnitude = np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))
    assert (np.abs(got - want) <= 4 * 2.0 ** -24 * magnitude).all()


def test_values_the_pieces_cannot_carry(hip):
    """Infinities, NaN and values next to the largest f32: the tiles they touch give what f32 arithmetic on the operands
    gives, the other tiles are not disturbed.  Rows below 2^-110 are carried like any other."""
    m, n, k = 1233, 1000, 700
    rng = np.random.default_rng(3)
    a, b = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(k, n)).astype(np.float32)
    clean = run(hip, m, n, k, "n", a, b)
    a[5, 17] = np.inf
    a[700, 3] = np.nan
    a[701] = 0.0
    a[701, 699] = 3.4e38  # rounds to infinity as bf16
    b[699, 4] = 0.5
    b[:, 999] *= np.float32(2.0 ** -118)
    a[1232] *= np.float32(2.0 ** -110)
    b[2, 130] = -np.inf
    got = run(hip, m, n, k, "n", a, b)
    with np.errstate(invalid="ignore", over="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        want = a64 @ b64
        magnitude = np.abs(a64) @ np.abs(b64)
    finite = np.isfinite(want) & (np.abs(want) < 3e38)
    assert (np.isnan(got) == np.isnan(want)).all()
    assert (got[np.isposinf(want)] == np.inf).all() and (got[np.isneginf(want)] == -np.inf).all()
    # sequential f32 sums: k roundings at most; below 2^-126 an f32 result is a multiple of 2^-149
    assert (np.abs(got[finite] - want[finite]) <= 2.0 ** -24 * k * magnitude[finite] + 2.0 ** -149 * k).all()
    assert (got[256:640, 256:900] == clean[256:640, 256:900]).all()


@pytest.mark.parametrize("layout", ["n", "t", "p"])
def test_marked_tiles_run_on_the_matrix_cores(hip, layout):
    """NaN throughout takes every tile to the f32 sums: about four times the ordinary time (a chain of multiply-adds per value
    took 130 to 300 times)."""
    m = n = k = 2048
    d_b, d_c = hip.DeviceBuffer.from_array(np.ones((k, n), np.float32)), hip.DeviceBuffer.from_array(np.zeros(m * n, np.float32))

    def best(value):
        d_a = hip.DeviceBuffer.from_array(np.full((m, k), value, np.float32))
        times = []
        for _ in range(5):
            start = time.perf_counter()
            if layout == "t":
                hip.gemm_f32_dev(m, n, k, 1.0, True, d_a, d_b, d_c)
            elif layout == "p":
                hip.gemm_prepacked_bias_act_f32_dev(m, n, k, 0, d_a, d_b, None, None, d_c)
            else:
                hip.gemm_bias_act_f32_dev(m, n, k, 0, d_a, d_b, None, None, d_c)
            hip.device_synchronize()
            times.append(time.perf_counter() - start)
        return min(times)

    assert hip.gemm_f32_split_plan(m, n, k, layout == "t", layout == "p")["served"]
    assert best(np.nan) <= 15 * best(1.0)


def test_the_shapes_above_run_on_the_split_kernels(hip):
    layouts = {"n": (False, False), "t": (True, False), "p": (False, True)}
    plans = {(shape, layout): hip.gemm_f32_split_plan(*shape, *layouts[layout]) for shape in SHAPES for layout in layouts}
    # (33 columns: the f32 kernels slice that reduction over workgroups unless B is prepacked)
    assert [case for case, plan in plans.items() if not plan["served"]] == [((4097, 33, 1003), "n"), ((4097, 33, 1003), "t")]
    plans = [plan for plan in plans.values() if plan["served"]]
    assert {plan["tile_rows"] for plan in plans} == {64, 96, 128, 160, 256}
    assert {plan["k_splits"] > 1 for plan in plans} == {False, True}
