"""What the library's host code asks of the runtime, with the runtime replaced by one that runs nothing (runtime_stub.cpp): no GPU."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

PRELUDE = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from spiraltorch_amd import _lib, hip
lib = _lib.load()
launches = ctypes.c_ulonglong.in_dll(stub, "stub_launches")
no_memory = ctypes.c_int.in_dll(stub, "stub_no_memory")
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("stub") / "libstub.so")
    subprocess.run(["hipcc", "-shared", "-fPIC", "-O1", "-x", "hip", "--offload-host-only", os.path.join(ROOT, "tests", "runtime_stub.cpp"), "-o", path], check=True)
    return path


def run(stub, body):
    done = subprocess.run([sys.executable, "-c", PRELUDE + body, stub], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout + done.stderr
    return done.stdout.split()


# few rows of all three bounds on what is packed, few columns, more rows than those; up to k = 1023 the general kernel needs no scratch
@pytest.mark.parametrize("m,n,k", [(3, 4001, 960), (8, 1001, 256), (33, 1001, 512), (17, 1953, 64), (500, 100, 512), (64, 127, 448)])
def test_products_go_on_without_room_for_a_packed_copy(stub, m, n, k):
    """A row-major bf16 B at odd boundaries is packed into scratch memory where that pays; without any to be had, the general kernel
    takes it as it is."""
    out = run(stub, f"""
for fail in (1, 0):
    no_memory.value, before = fail, launches.value
    hip.gemm_bf16_bias_act_dev({m}, {n}, {k}, 0, 1 << 20, 2 << 20, None, None, 3 << 20, None)
    print(launches.value - before)
""")
    assert out == ["1", "2"]


# around the bounds on what is copied for up to 64 rows, and on k
@pytest.mark.parametrize("m,n,k,launched", [(16, 663, 329, 2), (100, 1001, 300, 2), (64, 16384, 850, 2), (64, 16392, 65, 1), (64, 16384, 855, 1), (65, 40, 16383, 2),
                                            (3000, 40, 16385, 1), (20, 40, 63, 1),
                                            # one row of tiles: the general kernel where it reads a large B in less time than a pass over it takes
                                            (100, 51598, 218, 1), (92, 48000, 686, 1), (80, 33600, 736, 1), (80, 30000, 1001, 2), (128, 51598, 218, 2)])
def test_products_of_any_k_go_on_without_room_for_padded_copies(stub, m, n, k, launched):
    """A k that is no multiple of 64 is padded in scratch memory where that pays; without any to be had, the general kernel takes it as it
    is (a k it would cut over the chip needs scratch there too, as ever)."""
    out = run(stub, f"""
for fail in (1, 0) if {k} < 1024 else (0,):
    no_memory.value, before = fail, launches.value
    hip.gemm_bf16_bias_act_dev({m}, {n}, {k}, 0, 1 << 20, 2 << 20, None, None, 1 << 40, None)
    print(launches.value - before)
""")
    counts = [int(c) for c in out]
    if k < 1024:
        assert counts == [1, launched]
    else:  # padded: the pass and a product; not: slices of k and their sum
        assert counts[0] >= 2


@pytest.mark.parametrize("rows", [1, 64, 300])  # one value, and either side of the 256 KiB from which the pointer was looked at
def test_operands_in_device_memory_are_left_to_the_runtime(stub, rows):
    """A host call whose operand lies in device or managed memory (here: pages nobody may read) copies it with the runtime's copy."""
    out = run(stub, f"""
import mmap, numpy as np
libc = ctypes.CDLL(None)
libc.mmap.restype = ctypes.c_void_p
libc.mmap.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long]
count = {rows} * 256
closed = libc.mmap(None, 1 << 20, 0, mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS, -1, 0)
for name, value in (("stub_device_first", closed), ("stub_device_end", closed + (1 << 20))):
    ctypes.c_void_p.in_dll(stub, name).value = value
n = (1 << 22) // count + 1  # (a result that is not staged: no kernel writes one here)
rhs, out = np.ones(n, np.float32), np.zeros(count * n, np.float32)
status = lib.st_hip_gemm_f32(count, n, 1, 1.0, 0, closed, count, rhs.ctypes.data, n, out.ctypes.data, count * n)
print(status, ctypes.c_void_p.in_dll(stub, "stub_first_source").value == closed)
""")
    assert out == ["0", "True"]


def test_tensor_memory_goes_back_to_the_device_it_is_on(stub):
    """A tensor freed where another device is current (by a collector's thread, say) is not handed out there, and memory that is not a
    tensor's is not kept."""
    out = run(stub, """
device = ctypes.c_int.in_dll(stub, "stub_device")
def take():
    p = ctypes.c_void_p()
    assert lib.st_hip_tensor_malloc(ctypes.byref(p), 5000) == 0
    return p.value
first = take()
device.value = 1
lib.st_hip_tensor_free(first, 5000)
other = take()
device.value = 0
print(other != first, take() == first)
plain = ctypes.c_void_p()
lib.st_hip_malloc(ctypes.byref(plain), 5000)
lib.st_hip_tensor_free(plain, 5000)
second = take()
lib.st_hip_tensor_free(second, 5000)
print(take() == second)
""")
    assert out == ["True", "True", "True"]


def test_tensor_memory_is_freed_once(stub):
    """A second free of a tensor is an error, as the runtime's of any memory, and does not touch the block that is kept."""
    out = run(stub, """
import numpy as np
def take():
    p = ctypes.c_void_p()
    assert lib.st_hip_tensor_malloc(ctypes.byref(p), 5000) == 0
    return p.value
first, other = take(), take()
print(lib.st_hip_tensor_free(first, 5000) == 0, lib.st_hip_tensor_free(first, 5000) != 0, lib.st_hip_free(first) != 0)
host = np.zeros(16, np.uint8)
print(lib.st_hip_memcpy_h2d(first, host.ctypes.data, 16, None) != 0)
print(take() == first, take() not in (first, other))
print(lib.st_hip_tensor_free(first, 5000) == 0)
""")
    assert out == ["True"] * 7


def test_tensors_no_longer_used_make_room_for_those_that_are(stub):
    """All that is kept is of one size, and a program goes on with others: theirs are kept in its place, the longest idle go."""
    out = run(stub, """
frees = ctypes.c_ulonglong.in_dll(stub, "stub_frees")
def take(size):
    p = ctypes.c_void_p()
    assert lib.st_hip_tensor_malloc(ctypes.byref(p), size) == 0
    return p.value
MIB = 1 << 20
large = [take(8 * MIB) for _ in range(9)]
for p in large: lib.st_hip_tensor_free(p, 8 * MIB)
print(frees.value)  # the first of nine
small = [take(size) for size in (5000, 70000, 3 * MIB)]
for p, size in zip(small, (5000, 70000, 3 * MIB)): lib.st_hip_tensor_free(p, size)
print(frees.value)  # and the second
again = [take(size) for size in (5000, 70000, 3 * MIB)]
print(again == small, frees.value)
rest = [take(8 * MIB) for _ in range(7)]
print(sorted(rest) == sorted(large[2:]))
for p, size in zip(again, (5000, 70000, 3 * MIB)): lib.st_hip_tensor_free(p, size)
lib.st_hip_release_scratch(None)
print(frees.value)
""")
    assert out == ["1", "2", "True", "2", "True", "5"]


@pytest.mark.parametrize("call", ["hip.DeviceBuffer(20 << 20)", "hip.TensorBuffer(20 << 20)", "hip.TensorBuffer(3 << 20)",
                                  # a host call's operands, scratch for slices of k, a decoder's memory
                                  "hip.gemm_f32(2048, 8, 1024, np.ones(2 << 20, np.float32), np.ones(8 << 10, np.float32), np.ones(16 << 10, np.float32))",
                                  "hip.gemm_bf16_bias_act_dev(3000, 1000, 1000, 0, 1 << 20, 2 << 20, None, None, 3 << 20, None)",
                                  "hip.Decoder(256, 256, 4, 2, 1024, 1, 64, 1e-5, np.zeros(256 * 256 + 2 * (4 * 256 + 256 * 768 + 768 + 256 * 256 + 256 + 2 * (256 * 1024) + 1024 + 256) + 2 * 256 + 256 * 256 + 256, np.float32))"])
def test_allocations_take_the_room_that_freed_tensors_left(stub, call):
    out = run(stub, f"""
import numpy as np
frees = ctypes.c_ulonglong.in_dll(stub, "stub_frees")
used, most = (ctypes.c_ulonglong.in_dll(stub, "stub_memory_" + name) for name in ("used", "most"))
tensors = [hip.TensorBuffer(8 << 20) for _ in range(4)]
for tensor in tensors: tensor.free()
most.value = (32 << 20) + 1000
before = launches.value
try:
    {call}
    print("done")
except hip.HipErr as err:
    print("failed" if "hipMalloc" in str(err) or "OutOfMemory" in str(err) else "done")
print(frees.value >= 4, launches.value - before)
""")
    assert out[:2] == ["done", "True"], out
    if "bf16" in call:
        assert out[2] == "2"  # the padded copies and the product on them


def test_copies_past_the_end_of_device_memory_are_refused(stub):
    """A read that a kernel makes, and a tensor's upload, are refused where the runtime's copy refuses: no kernel is launched."""
    out = run(stub, """
import numpy as np
host, memory = np.zeros(9000, np.uint8), np.zeros(9000, np.uint8)
first = (memory.ctypes.data + 15) // 16 * 16
for name, value in (("stub_device_first", first), ("stub_device_end", first + 5000)):
    ctypes.c_void_p.in_dll(stub, name).value = value
def launched(call, *args):
    before = launches.value
    status = call(*args)
    return launches.value - before, status != 0
read = lambda at, bytes: launched(lib.st_hip_memcpy_d2h, host.ctypes.data, at, bytes, None)
send = lambda at, bytes: launched(lib.st_hip_tensor_upload, at, host.ctypes.data, bytes)
for at in (first, first + 4096):
    room = first + 5000 - at
    print(read(at, room)[0], read(at, room + 1) == (0, True), send(at, room)[0], send(at, room + 1) == (0, True))
""")
    assert out == ["1", "True", "1", "True"] * 2


def test_a_read_on_a_stream_of_another_device_is_left_to_the_runtime(stub):
    """The kernel would run there and read memory of the current device."""
    out = run(stub, """
import numpy as np
host, tensor, stream = np.zeros(4096, np.uint8), hip.TensorBuffer(4096), hip.Stream()
current, device = (ctypes.c_int.in_dll(stub, name) for name in ("stub_device", "stub_stream_device"))
for current.value, device.value in ((0, 0), (0, 1), (1, 0)):
    before = launches.value
    status = lib.st_hip_memcpy_d2h(host.ctypes.data, tensor.ptr, 4096, stream.ptr)
    print(launches.value - before)
print(status)
""")
    assert out == ["1", "0", "0", "0"]


def test_copies_past_the_end_of_a_tensor_are_refused(stub):
    """A tensor's block is larger than the tensor; what lies behind it is not the tensor's, now or when the block was another's."""
    out = run(stub, """
import numpy as np
host = np.zeros(20000, np.uint8)
p = ctypes.c_void_p()
for size in (8000, 5000, 6000):
    assert lib.st_hip_tensor_malloc(ctypes.byref(p), size) == 0
    first = p.value
    for at in (first, first + 4096, first + size - 1):
        room = first + size - at
        before = launches.value
        kept = (lib.st_hip_memcpy_h2d(at, host.ctypes.data, room, None), lib.st_hip_memset_zero(at, room, None))
        refused = [call != 0 for call in (
            lib.st_hip_tensor_upload(at, host.ctypes.data, room + 1), lib.st_hip_memcpy_h2d(at, host.ctypes.data, room + 1, None),
            lib.st_hip_memcpy_d2h(host.ctypes.data, at, room + 1, None), lib.st_hip_memset_zero(at, room + 1, None))]
        print(kept == (0, 0), all(refused), launches.value == before)
    before = launches.value
    print(lib.st_hip_tensor_upload(first, host.ctypes.data, size) == 0, launches.value == before + 1)
    lib.st_hip_tensor_free(first, size)
lib.st_hip_tensor_malloc(ctypes.byref(p), 5000)
lib.st_hip_free(p)
print(lib.st_hip_memcpy_h2d(p, host.ctypes.data, 6000, None) == 0)  # whatever is there next
""")
    assert out == ["True"] * len(out) and len(out) == 34


@pytest.mark.parametrize("batch,c_out,side,launched", [
    (64, 16, 28, 1), (65, 16, 28, 2), (48, 16, 36, 1), (49, 16, 36, 2), (128, 16, 20, 1), (129, 16, 20, 2), (128, 255, 7, 1), (129, 255, 7, 2), (64, 64, 29, 2), (256, 256, 7, 1), (257, 256, 7, 2),
    (100, 256, 28, 1), (4096, 511, 4, 2), (4096, 512, 4, 1), (8192, 512, 4, 1), (8193, 512, 4, 2), (16, 64, 90, 1), (16, 64, 91, 2), (32, 64, 57, 1), (32, 64, 58, 2), (33, 64, 44, 1), (33, 64, 45, 2),
    (32, 128, 64, 1), (32, 128, 65, 2), (33, 128, 50, 2), (48, 255, 36, 1), (48, 255, 37, 2), (48, 512, 1, 1), (49, 512, 1, 2), (1, 3, 1, 1), (65536, 16, 1, 2)])
def test_bias_gradients_of_many_images_are_spread_over_the_chip(stub, batch, c_out, side, launched):
    out = run(stub, f"""
for no_memory.value in (1, 0):
    before = launches.value
    hip.conv2d_grad_bias_f32_dev({batch}, 1, {side}, {side}, {c_out}, (1, 1), (1, 1), (0, 0), (1, 1), 1 << 20, 1.0, 2 << 20)
    print(launches.value - before)
""")
    assert out == ["1", str(launched)]  # in one without scratch memory


# planes much smaller than a workgroup's threads, weights of up to 64 KiB and beyond, and either side of each line of the rule
@pytest.mark.parametrize("batch,c_in,h,w,c_out,kernel,form", [
    (600, 512, 14, 14, 3, 3, "shared"), (600, 1000, 14, 14, 4, 3, "shared"), (512, 900, 12, 12, 4, 3, "shared"), (2048, 96, 7, 7, 3, 5, "shared"), (128, 512, 64, 64, 4, 3, "whole"),
    (127, 512, 64, 64, 4, 3, "shared"), (600, 47, 32, 32, 4, 3, "whole"), (1024, 64, 16, 32, 4, 3, "whole"), (1023, 64, 16, 32, 4, 3, "shared"), (5377, 113, 4, 7, 4, 7, "pixel"),
    (3924, 259, 8, 8, 4, 5, "pixel"), (1024, 500, 8, 11, 4, 3, "pixel"), (1024, 500, 9, 9, 4, 3, "shared"), (1024, 500, 16, 16, 4, 3, "shared"), (1024, 500, 13, 17, 4, 3, "pixel"),
    (1024, 500, 16, 19, 4, 3, "shared"), (1024, 455, 13, 17, 4, 3, "shared"), (64, 1025, 64, 64, 4, 3, "pixel"), (64, 1024, 64, 64, 4, 3, "shared")])
def test_convolutions_onto_few_channels_take_the_form_for_their_planes(stub, batch, c_in, h, w, c_out, kernel, form):
    out = run(stub, f"""
lds = ctypes.c_ulonglong.in_dll(stub, "stub_lds")
shape = ({batch}, {c_in}, {h}, {w}, {c_out}, ({kernel}, {kernel}), (1, 1), ({kernel // 2}, {kernel // 2}), (1, 1))
assert hip.conv2d_planned_kernel(*shape) == "direct"
hip.conv2d_bias_act_f32_dev(*shape, 0, 1 << 20, 2 << 20, None, 3 << 20)
print(lds.value)
""")
    weights = 4 * c_out * c_in * kernel * kernel
    assert int(out[0]) == {"pixel": 0, "whole": weights, "shared": weights + 4096 * c_out}[form]


@pytest.mark.parametrize("dilation,served", [(16383, True), (16384, False), (20000, False)])
def test_a_layer_whose_taps_are_too_far_apart_is_refused_whole(stub, dilation, served):
    """Forward and input gradient refuse the same layers, whichever kernel would run."""
    out = run(stub, f"""
pad = {dilation} - 20
shape = (32, 64, 56, 96, 64, (3, 3), (1, 1), (1, pad), (1, {dilation}))
assert hip.conv2d_output_hw(56, 96, *shape[5:]) == (56, 56)
def refused(call, *operands):
    try:
        call(*operands)
    except hip.HipErr:
        return True
    return False
for family in ("auto", "tile", "strip"):
    hip.conv2d_force_family(family)
    print(refused(hip.conv2d_bias_act_f32_dev, *shape, 0, 1 << 20, 2 << 20, None, 3 << 20), refused(hip.conv2d_grad_input_f32_dev, *shape, 1 << 20, 2 << 20, 3 << 20))
""")
    assert out == [str(not served)] * 6


def test_bf16_attention_launches_pass_their_check(stub):
    """Every grid the launchers of bf16 attention ask for passes the check made of it with the kernels' own decode."""
    out = run(stub, """
import itertools
calls = 0
for batch, heads, seq, dim, causal in itertools.product((1, 2, 3, 8), (1, 4, 7, 8), (1, 31, 32, 33, 64, 65, 128, 129, 500, 1000, 2048), (64, 128), (False, True)):
    hip.attention_bf16_dev(batch, heads, seq, dim, 0.125, causal, 1 << 20, 2 << 20, 3 << 20, 3 * heads * dim, 4 << 20, heads * dim)
    calls += 1
print(calls == launches.value)
""")
    assert out == ["True"]


@pytest.mark.parametrize("m,k,columns", [(3, 128, 7099), (16, 192, 9699), (17, 64, 7649), (40, 512, 18125), (16, 960, 7291), (40, 960, 10415)])
def test_how_many_columns_are_packed(stub, m, k, columns):
    """Few rows against a row-major bf16 B at odd boundaries: packed (two launches) up to so many columns, the general kernel beyond."""
    out = run(stub, f"""
for n in ({columns}, {columns} + 2):
    before = launches.value
    hip.gemm_bf16_bias_act_dev({m}, n, {k}, 0, 1 << 20, 2 << 20, None, None, 3 << 20, None)
    print(launches.value - before)
""")
    assert out[0] == "2" and out[1] == "1"
