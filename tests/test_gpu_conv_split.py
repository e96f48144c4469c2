"""f32 convolutions that run on the bf16 matrix cores as sums of three exact bf16 pieces, against float64."""
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# batch, c_in, h, w, c_out, kernel, stride, padding, dilation.  Pixels and channels one off the tiles (64, 128, 160, 256
# pixels, 32, 64, 128 channels), channel counts that are no multiple of 16, an odd number of steps, planes of which a tile
# holds several, strides, dilation, padding wider than the kernel's reach, one tap, a split of the reduction.
SHAPES = [
    (32, 64, 28, 28, 128, (3, 3), (1, 1), (1, 1), (1, 1)),
    (31, 64, 29, 27, 129, (3, 3), (1, 1), (1, 1), (1, 1)),
    (33, 33, 41, 47, 97, (3, 3), (1, 1), (1, 1), (1, 1)),
    (32, 250, 14, 14, 251, (3, 3), (1, 1), (1, 1), (1, 1)),
    (31, 512, 7, 7, 512, (3, 3), (1, 1), (1, 1), (1, 1)),
    (31, 513, 15, 13, 500, (1, 1), (1, 1), (0, 0), (1, 1)),
    (8, 48, 63, 61, 96, (5, 3), (2, 1), (2, 0), (1, 1)),
    (24, 80, 41, 40, 65, (3, 3), (1, 1), (2, 2), (2, 2)),
    (16, 64, 30, 31, 130, (3, 3), (1, 1), (4, 3), (1, 1)),
    (2, 512, 28, 28, 256, (3, 3), (1, 1), (1, 1), (1, 1)),
    (3, 40, 112, 113, 31, (7, 7), (1, 1), (3, 3), (1, 1)),
]


def forward64(case, x, w):
    batch, c_in, h, wd, c_out, kernel, stride, padding, dilation = case
    return torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), None, stride, padding, dilation).numpy()


def forward(hip, case, x, w, bias, activation=0):
    batch, c_in, h, wd, c_out, kernel, stride, padding, dilation = case
    oh, ow = hip.conv2d_output_hw(h, wd, kernel, stride, padding, dilation)
    n = batch * c_out * oh * ow
    d_out = hip.DeviceBuffer.from_array(np.full(n + 64, 7.5, np.float32))
    d_bias = None if bias is None else hip.DeviceBuffer.from_array(bias)
    d_x, d_w = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer.from_array(w)
    hip.conv2d_bias_act_f32_dev(*case, activation, d_x, d_w, d_bias, d_out)
    hip.device_synchronize()
    out = d_out.to_array(np.float32, n + 64)
    assert (out[n:] == 7.5).all(), "wrote past the end of the result"
    return out[:n].reshape(batch, c_out, oh, ow)


def check(got, product, want, terms):
    # One rounding (at most 2^-24 of the sum) per sixteen terms and a few at the end, independent of each other.  Leaving
    # out any one of the pieces costs 2^-18 of a product and fails this.
    bound = 2.0 ** -24 * np.sqrt(terms / 16 + 8) * np.sqrt(np.mean(product ** 2))
    assert np.sqrt(np.mean((got - want) ** 2)) <= bound
    assert np.abs(got - want).max() <= 8 * bound  # eight standard deviations


@pytest.mark.parametrize("case", SHAPES)
def test_forward_against_float64(hip, case):
    batch, c_in, h, wd, c_out, kernel = case[:6]
    rng = np.random.default_rng(sum(case[:5]))
    x = rng.normal(size=(batch, c_in, h, wd)).astype(np.float32)
    w = rng.normal(size=(c_out, c_in, *kernel)).astype(np.float32)
    bias = rng.normal(size=c_out).astype(np.float32)
    got = forward(hip, case, x, w, bias, 1)
    product = forward64(case, x, w)
    check(got, product, np.maximum(product + bias[None, :, None, None], 0.0), c_in * kernel[0] * kernel[1])


@pytest.mark.parametrize("case", [s for s in SHAPES if s[6] == (1, 1) and s[7][0] <= s[8][0] * (s[5][0] - 1)])
def test_grad_input_against_float64(hip, case):
    batch, c_in, h, wd, c_out, kernel, stride, padding, dilation = case
    oh, ow = hip.conv2d_output_hw(h, wd, kernel, stride, padding, dilation)
    rng = np.random.default_rng(sum(case[:5]) + 1)
    g = rng.normal(size=(batch, c_out, oh, ow)).astype(np.float32)
    w = rng.normal(size=(c_out, c_in, *kernel)).astype(np.float32)
    n = batch * c_in * h * wd
    d_gi = hip.DeviceBuffer.from_array(np.full(n + 64, 7.5, np.float32))
    d_g, d_w = hip.DeviceBuffer.from_array(g), hip.DeviceBuffer.from_array(w)
    hip.conv2d_grad_input_f32_dev(*case, d_g, d_w, d_gi)
    hip.device_synchronize()
    got = d_gi.to_array(np.float32, n + 64)
    assert (got[n:] == 7.5).all(), "wrote past the end of the result"
    want = torch.nn.functional.conv_transpose2d(torch.from_numpy(g).double(), torch.from_numpy(w).double(), None, stride, padding, 0, 1, dilation)
    want = want.numpy()
    check(got[:n].reshape(batch, c_in, h, wd), want, want, c_out * kernel[0] * kernel[1])


def test_finite_operands_whose_products_overflow(hip):
    case = (32, 64, 28, 28, 128, (3, 3), (1, 1), (1, 1), (1, 1))
    rng = np.random.default_rng(4)
    x = rng.normal(size=(32, 64, 28, 28)).astype(np.float32)
    w = np.full((128, 64, 3, 3), 1.3e25, np.float32)
    w[::2] *= -1.0
    x[3] = rng.uniform(1e25, 2e25, (64, 28, 28))
    for activation in (0, 1):
        got = forward(hip, case, x, w, None, activation)
        assert (got[3, 1::2] == np.inf).all() and (got[3, ::2] == (0.0 if activation else -np.inf)).all()
        others = np.arange(32) != 3
        want = forward64(case, x[others], w)
        want = np.maximum(want, 0.0) if activation else want
        # f32 sums of 576 terms, their roundings in quadrature, eight standard deviations
        assert np.abs(got[others] - want).max() <= 8 * 2.0 ** -24 * np.sqrt(576) * 24 * 1.3e25


def test_small_values_beside_ordinary_ones(hip):
    case = (32, 64, 28, 28, 128, (3, 3), (1, 1), (1, 1), (1, 1))
    rng = np.random.default_rng(5)
    x = rng.normal(size=(32, 64, 28, 28)).astype(np.float32)
    x[:, 5] = (rng.normal(size=(32, 28, 28)) * 1e-37).astype(np.float32)  # subnormal ones among them
    w = np.zeros((128, 64, 3, 3), np.float32)
    w[:, 5] = (rng.normal(size=(128, 3, 3)) * 1e20).astype(np.float32)
    got, want = forward(hip, case, x, w, None), forward64(case, x, w)
    magnitude = forward64(case, np.abs(x), np.abs(w))
    # nine products, of each at most 2^-24 left out, their sums rounded at most nine times
    assert (np.abs(got - want) <= 10 * 2.0 ** -24 * magnitude).all()


def test_values_the_pieces_cannot_carry(hip):
    case = (32, 64, 28, 28, 128, (3, 3), (1, 1), (1, 1), (1, 1))
    rng = np.random.default_rng(3)
    x = rng.normal(size=(32, 64, 28, 28)).astype(np.float32)
    w = rng.normal(size=(128, 64, 3, 3)).astype(np.float32)
    plain = forward(hip, case, x, w, None)
    x[1, 5, 10, 10] = np.inf
    x[2, 60, 27, 27] = np.nan
    x[3, 0, 0, 0] = 1.5 * 2.0 ** 127
    x[4] *= np.float32(2.0 ** -120)  # a whole image below 2^-110, partly subnormal
    x[5, :, :14] = 0.0
    x[6, 7, 3, 3] = 2.0 ** -130  # one small value among ordinary ones
    w[9] *= np.float32(2.0 ** -115)
    got = forward(hip, case, x, w, None)
    with np.errstate(all="ignore"):
        want = forward64(case, x, w)
    finite = np.abs(want) <= np.finfo(np.float32).max
    assert (np.isfinite(got) == finite).all()
    assert (np.isnan(got) == np.isnan(want)).all()
    for image in range(8):
        for channels in (np.arange(128) != 9, np.arange(128) == 9):
            ok = finite[image, channels]
            scale = np.sqrt(np.mean(want[image, channels][ok & (np.abs(want[image, channels]) < 1e30)] ** 2))
            # a plain f32 summation of 576 terms: their rounding errors in quadrature, eight standard deviations
            bound = 8 * 2.0 ** -24 * np.sqrt(576) * scale + 576 * 2.0 ** -149
            diff = np.abs(got[image, channels][ok] - want[image, channels][ok])
            assert (diff <= np.maximum(bound, 2.0 ** -20 * np.abs(want[image, channels][ok]))).all(), image
    # images and channels without such values: both runs keep to the bound above, the results' rms is 24
    untouched, keep = np.arange(32) >= 8, np.arange(128) != 9
    assert np.abs(got[untouched][:, keep] - plain[untouched][:, keep]).max() <= 8 * 2.0 ** -24 * np.sqrt(576) * 24


def test_marked_tiles_run_on_the_matrix_cores(hip):
    """NaN throughout takes every tile to the f32 sums: four to five times the ordinary time (a chain of multiply-adds per
    value took 65 to 100 times)."""
    case = (32, 256, 14, 14, 256, (3, 3), (1, 1), (1, 1), (1, 1))
    d_w, d_out = hip.DeviceBuffer.from_array(np.ones((256, 256, 3, 3), np.float32)), hip.DeviceBuffer.from_array(np.zeros(32 * 256 * 196, np.float32))

    def best(value):
        d_x = hip.DeviceBuffer.from_array(np.full((32, 256, 14, 14), value, np.float32))
        times = []
        for _ in range(5):
            start = time.perf_counter()
            hip.conv2d_bias_act_f32_dev(*case, 0, d_x, d_w, None, d_out)
            hip.device_synchronize()
            times.append(time.perf_counter() - start)
        return min(times)

    assert best(np.nan) <= 15 * best(1.0)


def test_the_shapes_above_run_on_the_split_kernels(hip):
    plans = [hip.conv2d_f32_split_plan(*case) for case in SHAPES]
    assert all(plan["served"] for plan in plans)
    assert {plan["tile_channels"] for plan in plans} == {32, 64, 128} and {plan["k_splits"] > 1 for plan in plans} == {False, True}
    assert sum(hip.conv2d_f32_split_plan(*case, direction="grad_input")["served"] for case in SHAPES) >= 7
    hip.conv2d_force_family("tile")
    try:
        assert not any(hip.conv2d_f32_split_plan(*case)["served"] for case in SHAPES)
    finally:
        hip.conv2d_force_family("auto")
