"""What the host-slice calls move through pinned memory, and the finite check's words: every byte, at the edges of pieces, from
several threads at once."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def outer(hip, column, row):
    """column · row as a host-slice product of one term: exact, every operand and result byte moved."""
    out = np.full(column.size * row.size, 7.5, np.float32)
    hip.gemm_f32(column.size, row.size, 1, column, row, out)
    return out.reshape(column.size, row.size)


# around a 16 KiB piece of the result, a 256 KiB piece of an operand, and what is no multiple of sixteen bytes
@pytest.mark.parametrize("m,n", [(1, 1), (3, 1), (1, 4095), (1, 4096), (1, 4097), (5, 819), (65536, 1), (65537, 1), (70001, 1), (131, 1021),
                                 (1024, 1024), (2049, 2051)])
def test_every_byte_arrives(hip, m, n):
    rng = np.random.default_rng(m + n)
    column, row = rng.integers(-999, 999, m).astype(np.float32), rng.integers(-999, 999, n).astype(np.float32)
    assert (outer(hip, column, row) == column[:, None] * row[None, :]).all()


# around the ring a result goes through (2 MiB in four quarters), several rounds of it, and the size that goes past it
@pytest.mark.parametrize("count", [(1 << 19) - 1, 1 << 19, (1 << 19) + 1, (1 << 19) + (1 << 17) + 5, 3 * (1 << 19) - 4097, (1 << 22) - 1, 1 << 22,
                                   (1 << 22) + 1])
def test_every_byte_of_results_larger_than_the_ring(hip, count):
    row = np.random.default_rng(count).integers(-(1 << 20), 1 << 20, count).astype(np.float32)
    assert (outer(hip, np.float32([-1.0]), row)[0] == -row).all()


def test_large_calls_do_not_pin_their_memory_anew(hip):
    """Operands and results of 16 MiB, from one thread and from four at once: what the first calls have pinned serves the others."""
    size = 2048
    a, b, bias = np.ones((size, size), np.float32), np.ones((size, size), np.float32), np.ones(size, np.float32)

    def work(calls):
        out = np.zeros(size * size, np.float32)
        for _ in range(calls):
            hip.gemm_bias_activation_f32(size, size, size, hip.GemmActivation.Relu, a, b, bias, None, out)

    hip.release_scratch()
    for threads in (1, 4):
        def together(calls):
            workers = [threading.Thread(target=work, args=(calls,)) for _ in range(threads)]
            for t in workers:
                t.start()
            for t in workers:
                t.join()

        together(4)
        _, before = hip.pinned_memory_counters()
        together(6)
        held, after = hip.pinned_memory_counters()
        assert held <= 64 << 20
        # (four threads may never have held the few buffers of a call at the same moment before)
        assert after - before <= (0 if threads == 1 else 8)
    hip.release_scratch()
    assert hip.pinned_memory_counters()[0] == 0


def test_pinned_operands_and_results(hip):
    """Host memory that is pinned already is copied from and to directly."""
    runtime = ctypes.CDLL("libamdhip64.so.7")  # the one the library is linked with
    m, n = 600, 700
    rng = np.random.default_rng(1)
    blocks, arrays = [], []
    for size in (m, n, m * n):
        block = ctypes.c_void_p()
        assert runtime.hipHostMalloc(ctypes.byref(block), ctypes.c_size_t(size * 4), ctypes.c_uint(0)) == 0
        blocks.append(block)
        arrays.append(np.ctypeslib.as_array(ctypes.cast(block, ctypes.POINTER(ctypes.c_float)), (size,)))
    arrays[0][:], arrays[1][:] = rng.integers(-99, 99, m), rng.integers(-99, 99, n)
    hip.gemm_f32(m, n, 1, *arrays)
    assert (arrays[2].reshape(m, n) == arrays[0][:, None] * arrays[1][None, :]).all()
    del arrays
    for block in blocks:
        assert runtime.hipHostFree(block) == 0


def test_calls_from_several_threads_keep_their_bytes(hip):
    wrong = []

    def work(seed):
        rng = np.random.default_rng(seed)
        for _ in range(20):
            m, n = int(rng.integers(1, 700)), int(rng.integers(1, 700))
            column, row = rng.integers(-999, 999, m).astype(np.float32), rng.integers(-999, 999, n).astype(np.float32)
            if not (outer(hip, column, row) == column[:, None] * row[None, :]).all():
                wrong.append((seed, m, n))
            data = rng.normal(size=m * n).astype(np.float32)
            data[m * n // 2] = np.nan
            d_data = hip.DeviceBuffer.from_array(data)
            if hip.count_nonfinite_f32_dev(m * n, d_data)[:2] != (1, m * n // 2):
                wrong.append((seed, m, n, "count"))

    threads = [threading.Thread(target=work, args=(seed,)) for seed in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == []


@pytest.mark.parametrize("count", [1, 3, 4, 5, 255, 2047, 2048, 2049, 8193, (1 << 20) + 3, 512 * 2048 * 3 + 1])
def test_count_nonfinite(hip, count):
    """Counts and first indices at both ends, at any alignment, with infinities and NaN."""
    data = np.ones(count + 1, np.float32)
    d = hip.DeviceBuffer.from_array(data)
    for shift in (0, 1):
        assert hip.count_nonfinite_f32_dev(count, d.at(4 * shift)) == (0, 0, 0.0)
    for places in ({0}, {count - 1}, {0, count // 2, count - 1}):  # (fewer where they coincide)
        bad = data.copy()
        for i, place in enumerate(sorted(places)):
            bad[1 + place] = (np.inf, -np.inf, np.nan)[i]
        d_bad = hip.DeviceBuffer.from_array(bad)
        found, first, value = hip.count_nonfinite_f32_dev(count, d_bad.at(4))
        assert (found, first) == (len(places), min(places)) and value == np.inf


def test_copies_after_the_kept_memory_was_freed(hip):
    column, row = np.arange(1, 300, dtype=np.float32), np.arange(1, 200, dtype=np.float32)
    for _ in range(3):
        assert (outer(hip, column, row) == column[:, None] * row[None, :]).all()
        hip.release_scratch()


@pytest.mark.parametrize("size", [1, 7, 8, 9, 4095, 4096, 4097, 16383, 16384, 16385, 100003, (1 << 19) - 1, 1 << 19, (1 << 19) + 1, (1 << 21) - 3, 1 << 21, (1 << 21) + 5])
def test_every_byte_of_a_tensor_up_and_down(hip, size):
    """Around a workgroup's part of an upload, a piece of a read, what is staged up and down, and what is no multiple of eight bytes."""
    data = np.random.default_rng(size).integers(0, 256, size).astype(np.uint8)
    for kind in (hip.TensorBuffer, hip.DeviceBuffer):
        d = kind.from_array(data)
        assert (d.to_array(np.uint8, size) == data).all()
        if size > 5000:  # from the middle, on a 16-byte boundary and off it
            for first in (4096, 4099):
                out = np.empty(size - first, np.uint8)
                status = __import__("spiraltorch_amd._lib", fromlist=["load"]).load().st_hip_memcpy_d2h(
                    ctypes.c_void_p(out.ctypes.data), ctypes.c_void_p(d.at(first)), out.nbytes, None)
                assert status == 0 and (out == data[first:]).all()


def test_tensor_memory_taken_over_while_its_last_use_is_queued(hip):
    """A tensor is freed with kernels on it still queued, and its memory goes to the next one, whose values are uploaded at once."""
    n = 128 * 1024  # half a MiB: staged
    before = hip.DeviceBuffer.from_array(np.arange(n, dtype=np.float32))
    outs = [hip.DeviceBuffer(n * 4) for _ in range(8)]
    busy = hip.DeviceBuffer.from_array(np.zeros((2048, 2048), np.float32))
    result = hip.DeviceBuffer(2048 * 2048 * 4)
    addresses, source = set(), np.empty(n, np.float32)
    for i, out in enumerate(outs):
        source[:] = i + 1.0
        tensor = hip.TensorBuffer.from_array(source)
        source[:] = -77.0  # the call has taken its copy
        addresses.add(tensor.ptr.value)
        hip.gemm_f32_dev(2048, 2048, 2048, 1.0, False, busy, busy, result)  # the reads below are queued behind this
        hip.scale_f32_dev(n, tensor, 2.0, out)
        tensor.free()
    assert len(addresses) < len(outs)
    for i, out in enumerate(outs):
        assert (out.to_array(np.float32, n) == 2.0 * (i + 1.0)).all(), i
    assert (before.to_array(np.float32, n) == np.arange(n)).all()


def test_tensors_from_several_threads_keep_their_values(hip):
    import spiraltorch_amd as st
    wrong = []

    def work(seed):
        rng = np.random.default_rng(seed)
        for _ in range(40):
            rows, cols = int(rng.integers(1, 300)), int(rng.integers(1, 300))
            x = rng.integers(-99, 99, (rows, cols)).astype(np.float32)
            y = st.Tensor.from_numpy(x).scale(2.0).scale(0.25)
            if not (y.numpy() == x * 0.5).all():
                wrong.append((seed, rows, cols))

    threads = [threading.Thread(target=work, args=(seed,)) for seed in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == []
    hip.release_scratch()
    assert hip.pinned_memory_counters()[0] == 0


# operands that go up together, and one value past what does, first, last and both; parts of 4 KiB cut short
@pytest.mark.parametrize("m,n", [(1023, 1025), (32767, 3), (32768, 5), (32769, 5), (3, 32768), (5, 32769), (32768, 32), (32769, 33)])
def test_operands_that_go_up_together(hip, m, n):
    rng = np.random.default_rng(m + n)
    column, row = rng.integers(-999, 999, m).astype(np.float32), rng.integers(-999, 999, n).astype(np.float32)
    bias = rng.integers(-999, 999, n).astype(np.float32)
    residual = rng.integers(-999, 999, m * n).astype(np.float32)
    out = np.full(m * n, 7.5, np.float32)
    hip.gemm_bias_activation_f32(m, n, 1, hip.GemmActivation.Relu, column, row, bias, residual, out)
    want = column[:, None] * row[None, :] + bias + residual.reshape(m, n)
    assert (out.reshape(m, n) == np.maximum(want, 0.0)).all()
