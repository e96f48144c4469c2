"""bf16 products of few rows on small tiles with k split inside the workgroup (gemm_bf16_small.hip)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 16, 64), (33, 8, 128), (31, 40, 64),          # one wavefront with work, tiles that hang over both ends
    (117, 512, 512), (117, 1536, 512), (65, 504, 576),  # a stage a wavefront; nine k-tiles over eight wavefronts
    (40, 500, 512), (40, 257, 1024),                  # rows of B off 16-byte boundaries (packed first); an odd width
    (9, 3500, 2048), (9, 3412, 2048), (33, 4884, 2048),  # row-major: just beyond and within what is packed, of few and more rows
    (3, 7099, 128), (17, 7649, 64), (40, 18125, 512),  # the most columns that are packed
    (117, 512, 2048), (64, 768, 3136),                # several stages a wavefront, an uneven last share
    (1024, 512, 2048), (600, 1000, 448), (2048, 300, 640),  # 64×64 tiles; groups of eight row tiles, a ragged last one
    (545, 72, 256),                                   # a grid that eight does not divide, a group of one or two row tiles
])
def test_small_tiles(hip, m, n, k):
    """Both layouts of B, plain and with scale-free bias + residual + GELU into both outputs, against float64.  The bound: the
    products are exact in f32, so a sum of k of them is off by at most k roundings of the sum of magnitudes."""
    from spiraltorch_amd import inputs
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a, b = inputs.to_bf16(rng.normal(size=m * k).astype(np.float32)), inputs.to_bf16(rng.normal(size=k * n).astype(np.float32))
    a64, b64 = inputs.from_bf16(a).reshape(m, k).astype(np.float64), inputs.from_bf16(b).reshape(k, n).astype(np.float64)
    bias, res = rng.normal(size=n).astype(np.float32), rng.normal(size=(m, n)).astype(np.float32)
    d_a, d_bias, d_res = (hip.DeviceBuffer.from_array(v) for v in (a, bias, res))
    d_b, d_packed = hip.DeviceBuffer.from_array(b), hip.DeviceBuffer.from_array(np.ascontiguousarray(b.reshape(k, n).T))
    plain, bound = a64 @ b64, k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)) + 1e-30
    pre = plain + bias + res
    gelu = 0.5 * pre * (1.0 + np.tanh(0.7978846 * (pre + 0.044715 * pre ** 3)))
    seen = {}
    for packed in (True, False):
        call = hip.gemm_bf16_prepacked_bias_act_dev if packed else hip.gemm_bf16_bias_act_dev
        operand = d_packed if packed else d_b
        guard = 64
        d32, d16 = hip.DeviceBuffer((m * n + guard) * 4), hip.DeviceBuffer((m * n + guard) * 2)
        d32.zero()
        call(m, n, k, 0, d_a, operand, None, None, d32, None)
        hip.device_synchronize()
        got = d32.to_array(np.float32, m * n + guard)
        assert (got[m * n:] == 0).all(), "stores past the result"
        assert (np.abs(got[:m * n].reshape(m, n) - plain) <= bound).all(), f"packed={packed}"
        call(m, n, k, int(hip.GemmActivation.Gelu), d_a, operand, d_bias, d_res, d32, d16)
        hip.device_synchronize()
        got32 = d32.to_array(np.float32, m * n + guard)[:m * n].reshape(m, n)
        # GELU's slope is at most 1.13; its own evaluation and the two additions add a few roundings of the value
        assert (np.abs(got32 - gelu) <= 1.13 * bound + 2e-6 * (np.abs(pre) + 1.0)).all(), f"epilogue packed={packed}"
        assert (d16.to_array(np.uint16, m * n + guard)[:m * n] == inputs.to_bf16(got32.ravel())).all()
        seen[packed] = (got[:m * n], got32)
    if m > 64 or k <= 1024:  # (a row-major B of few rows and a long k takes the skinny kernel)
        assert all((x == y).all() for x, y in zip(seen[True], seen[False])), "both layouts add in the same order"


def test_small_tiles_of_non_finite_operands(hip):
    """Infinities and NaN reach the rows they belong to, and no other: rows past the end of a tile are not mixed in."""
    from spiraltorch_amd import inputs
    m, n, k = 45, 200, 512
    rng = np.random.default_rng(5)
    a, b = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(n, k)).astype(np.float32)
    a[7, 100], a[44, 3] = np.inf, np.nan
    d_a, d_b = hip.DeviceBuffer.from_array(inputs.to_bf16(a.ravel())), hip.DeviceBuffer.from_array(inputs.to_bf16(b.ravel()))
    out = hip.DeviceBuffer(m * n * 4)
    hip.gemm_bf16_prepacked_bias_act_dev(m, n, k, 0, d_a, d_b, None, None, out, None)
    hip.device_synchronize()
    got = out.to_array(np.float32, m * n).reshape(m, n)
    assert np.isinf(got[7]).all() and np.isnan(got[44]).all()
    assert np.isfinite(np.delete(got, (7, 44), axis=0)).all()


@pytest.mark.parametrize("m,n,k,layouts,behind", [
    (1024, 49408, 64, "pr", 256), (2048, 24832, 128, "r", 256),   # 772 and 776 tiles of 256×256, B as it is
    (1024, 50257, 64, "p", 1105), (2047, 24700, 192, "pr", 124),  # columns off every boundary, ragged rows; a row-major B packed first
    # a last round of a few tiles as well, but in tiles of 256×128 throughout
    (1024, 16600, 64, "p", 0), (1024, 16641, 192, "pr", 0), (1000, 16640, 128, "pr", 0), (2049, 8064, 64, "pr", 0), (300, 33024, 64, "p", 0),
])
def test_columns_behind_the_full_rounds(hip, m, n, k, layouts, behind):
    """A last round of a few 256×256 tiles runs as 128×128 tiles in a launch of its own: every column against float64 (the bound
    as above), and the columns of the full rounds bit for bit what a product of those alone gives."""
    from spiraltorch_amd import inputs
    assert ("columns_behind" in hip.gemm_bf16_routes(m, n, k)) == (behind > 0)
    whole = n - behind
    rng = np.random.default_rng(m + n + k)
    a, b = inputs.to_bf16(rng.normal(size=m * k).astype(np.float32)), inputs.to_bf16(rng.normal(size=n * k).astype(np.float32))
    bias = rng.normal(size=n).astype(np.float32)
    a64, b64 = inputs.from_bf16(a).reshape(m, k).astype(np.float64), inputs.from_bf16(b).reshape(n, k).astype(np.float64)
    want, bound = a64 @ b64.T + bias, k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64).T + np.abs(bias))
    d_a, d_bias, d_p = hip.DeviceBuffer.from_array(a), hip.DeviceBuffer.from_array(bias), hip.DeviceBuffer.from_array(b)
    d_r = hip.DeviceBuffer.from_array(np.ascontiguousarray(b.reshape(n, k).T))
    d32, d16 = hip.DeviceBuffer((m * n + 64) * 4), hip.DeviceBuffer(m * n * 2)
    bits = []
    if behind:
        assert not hip.gemm_bf16_routes(m, whole, k) and hip.gemm_bf16_tile_plan(m, whole, k)["tile_cols"] == 256
        hip.gemm_bf16_prepacked_bias_act_dev(m, whole, k, 0, d_a, d_p, d_bias, None, d32, d16)
        hip.device_synchronize()
        first = d32.to_array(np.float32, m * whole).reshape(m, whole)
    for layout in layouts:
        d32.zero()
        call, operand = (hip.gemm_bf16_prepacked_bias_act_dev, d_p) if layout == "p" else (hip.gemm_bf16_bias_act_dev, d_r)
        call(m, n, k, 0, d_a, operand, d_bias, None, d32, d16)
        hip.device_synchronize()
        got = d32.to_array(np.float32, m * n + 64)
        assert (got[m * n:] == 0).all()
        bits.append(got[:m * n].reshape(m, n))
        assert (np.abs(bits[-1] - want) <= bound).all(), layout
        assert (d16.to_array(np.uint16, m * n) == inputs.to_bf16(got[:m * n])).all()
        if behind:
            assert (bits[-1][:, :whole] == first).all(), layout
    assert all((x == bits[0]).all() for x in bits)
