"""Row softmax with the row in the registers of one workgroup: rows at the edges of the kernel's piece counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# pieces of 2048 values: 4, 8, 16, 20 and 25 of them, one value around each, and the 1024-thread kernel beyond
@pytest.mark.parametrize("cols", [4097, 4099, 8191, 8192, 8193, 16384, 16387, 32768, 32770, 40960, 40961, 51199, 51200, 51201, 65535, 65536])
@pytest.mark.parametrize("in_place", [False, True])
def test_against_float64(hip, cols, in_place):
    rng = np.random.default_rng(cols)
    x = rng.normal(size=(5, cols)).astype(np.float32) * 3
    x[0, -1] = 90.0  # the last value decides the row
    x[1, ::2] = np.nan  # skipped
    x[2, cols // 3:] = -np.inf
    x[3] = np.nan
    x[3, cols - 2:] = -np.inf  # no usable sum: one at the first entry that holds the maximum
    x[4, [cols // 2, cols - 1]] = np.inf
    d_x = hip.DeviceBuffer.from_array(x)
    d_y = d_x if in_place else hip.DeviceBuffer.from_array(np.full(x.size + 64, 7.5, np.float32))
    hip.row_softmax_f32_dev(5, cols, d_x, d_y)
    hip.device_synchronize()
    if in_place:
        got = d_y.to_array(np.float32, x.size).reshape(5, cols)
    else:
        got = d_y.to_array(np.float32, x.size + 64)
        assert (got[x.size:] == 7.5).all(), "wrote past the end of the result"
        got = got[:x.size].reshape(5, cols)
    usable = np.where(np.isnan(x[:3]), -np.inf, x[:3]).astype(np.float64)
    e = np.exp(usable - usable.max(axis=1, keepdims=True))
    want = e / e.sum(axis=1, keepdims=True)
    # an exponent of up to 104 is rounded by half an ulp of 2^-17 before the exponential: 2^-18 relative, 2^-149 where it underflows
    assert (np.abs(got[:3] - want) <= 2.0 ** -17 * want + 2.0 ** -120).all()
    assert got[3].sum() == 1.0 and got[3, cols - 2] == 1.0
    assert got[4].sum() == 1.0 and got[4, cols // 2] == 1.0


@pytest.mark.parametrize("rows,cols", [(800, 50257), (8200, 5001), (1024, 65536)])  # beyond 128 MiB, 128 MiB, and 192 MiB of values
@pytest.mark.parametrize("in_place", [False, True])
def test_what_passes_the_cache_by_gives_the_same_bits(hip, rows, cols, in_place):
    few = np.random.default_rng(cols).normal(size=(7, cols)).astype(np.float32) * 3
    d_few, d_want = hip.DeviceBuffer.from_array(few), hip.DeviceBuffer(few.nbytes)
    hip.row_softmax_f32_dev(7, cols, d_few, d_want)
    order = np.arange(rows) % 7
    d_x = hip.DeviceBuffer.from_array(few[order])
    d_y = d_x if in_place else hip.DeviceBuffer(rows * cols * 4)
    hip.row_softmax_f32_dev(rows, cols, d_x, d_y)
    hip.device_synchronize()
    want = d_want.to_array(np.uint32, few.size).reshape(7, cols)
    assert (d_y.to_array(np.uint32, rows * cols).reshape(rows, cols) == want[order]).all()
