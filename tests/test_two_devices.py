"""What the launchers keep per device, on a stand-in runtime of two devices (host/two_devices.cpp; no GPU, no kernel runs):
each case is a program of its own, which loads the stand-in ahead of the library."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PROGRAM = r"""
import ctypes as C, sys
rt = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
from et_amd._lib import check, lib
L = lib()

def buf(n):  # device memory that no kernel touches
    p = C.c_void_p()
    check(L.et_malloc(C.byref(p), n))
    return p

def stream(device):
    s = C.c_void_p()
    rt.two_devices_stream(device, C.byref(s))
    return s

def launches():
    out = []
    for i in range(rt.two_devices_launches()):
        d, b, lds = C.c_int(), C.c_uint(), C.c_uint()
        rt.two_devices_launch(i, C.byref(d), C.byref(b), C.byref(lds))
        out.append((d.value, b.value, lds.value))
    return out

def plan(K, N, sparsity):
    rp = np.zeros(N // 16 + 1, np.int32)
    ro = np.zeros((N // 16) * (K // 16), np.int32)
    n = L.et_gen_sparse_tile_mat(N, K, sparsity, 1, rp.ctypes.data, ro.ctypes.data)
    data, bias = np.zeros(n * 256, np.uint16), np.zeros(N, np.uint16)
    p = C.c_void_p()
    check(L.et_tile_plan_create(C.byref(p), K, N, n, data.ctypes.data, rp.ctypes.data, ro.ctypes.data, bias.ctypes.data))
    return p

x = buf(1 << 20)
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler here")
    so = str(tmp_path_factory.mktemp("host") / "two_devices.so")
    res = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fPIC", "-shared", "-pthread", "-o", so,
                          os.path.join(HERE, "host", "two_devices.cpp")], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return so


def run(runtime, body):
    res = subprocess.run([sys.executable, "-c", PROGRAM + body, runtime, ROOT], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, (res.stdout + res.stderr)[-3000:]


ATTENTION = {
    "padded": "L.et_OTF_attention(x, x, x, x, None, 1024, 768, 12, 1, None, 1.0, s)",
    "masked": "L.et_OTF_attention(x, x, x, x, x, 1000, 768, 12, 1, None, 1.0, s)",
    "packed": "L.et_OTF_attention_varlen(x, x, x, x, None, x, 1024, 768, 12, 1, 1.0, s)",
    "packed masked": "L.et_OTF_attention_varlen(x, x, x, x, x, x, 1024, 768, 12, 1, 1.0, s)",
}


@pytest.mark.parametrize("form", ATTENTION)
def test_attention_above_64_kb_of_lds_on_a_second_device(runtime, form):
    """two key groups take 80 KB: every device needs the opt-in"""
    run(runtime, f"""
s = None
for device in (0, 1, 0):
    rt.hipSetDevice(device)
    rt.two_devices_clear()
    check({ATTENTION[form]})
    ls = launches()
    assert len(ls) == 1 and ls[0][0] == device and ls[0][2] > 64 * 1024, ls
""")
