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


# short rows: the edges of a wavefront's pieces (by values up to 128, by fours beyond), of 512, 1024 and 2048 values, and of the workgroup's two pieces
@pytest.mark.parametrize("cols", [1, 3, 5, 63, 64, 65, 127, 128, 129, 130, 511, 513, 1022, 1024, 1025, 2045, 2047, 2048, 2049, 2051, 4095, 4096])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_rows_of_any_length_at_any_boundary(hip, cols, offset):
    rng = np.random.default_rng(cols * 4 + offset)
    x = rng.normal(size=(6, cols)).astype(np.float32) * 3
    x[1, -1] = 60.0  # the last value decides the row
    x[2, 1::2] = np.nan  # skipped
    x[3, :] = np.nan  # zeros
    x[4, 0::2] = -np.inf
    x[5, :] = -np.inf  # no usable sum: one at the first entry that holds the maximum
    host = np.concatenate([np.zeros(offset, np.float32), x.reshape(-1)])
    d_x, d_y = hip.DeviceBuffer.from_array(host), hip.DeviceBuffer.from_array(np.full(x.size + 64, 7.5, np.float32))
    hip.row_softmax_f32_dev(6, cols, d_x.ptr.value + 4 * offset, d_y.ptr.value + 4 * offset)
    hip.device_synchronize()
    got = d_y.to_array(np.float32, x.size + 64)
    assert (got[:offset] == 7.5).all() and (got[offset + x.size:] == 7.5).all(), "wrote outside the result"
    got = got[offset:offset + x.size].reshape(6, cols)
    want = np.zeros((6, cols))
    for r in range(6):
        usable = np.where(np.isnan(x[r]), -np.inf, x[r]).astype(np.float64)
        if np.isfinite(usable.max()):
            e = np.exp(usable - usable.max())
            want[r] = e / e.sum()
        elif not np.isnan(x[r]).all():
            want[r, int(np.flatnonzero(~np.isnan(x[r]))[0])] = 1.0
    # an exponent of up to 75 is rounded by half an ulp of 2^-17 before the exponential: 2^-18 relative, 2^-149 where it underflows
    assert (np.abs(got - want) <= 2.0 ** -17 * want + 2.0 ** -120).all()
