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
