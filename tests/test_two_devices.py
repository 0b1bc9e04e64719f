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

def flow(rows):
    f = C.c_void_p()
    plans = [plan(768, 768, 0.8) for _ in range(4)] + [plan(768, 3072, 0.8), plan(3072, 768, 0.8)]
    check(L.et_layer_flow_create(C.byref(f), *plans, rows, 12, 1))
    assert f.value
    return f

x, y = buf(1 << 20), buf(1 << 20)
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


OTHER_STREAM = {
    "attention": "[L.et_OTF_attention(x, x, x, x, None, 1024, 768, 12, 1, None, 1.0, s)]",
    "packed attention": "[L.et_OTF_attention_varlen(x, x, x, x, x, x, 1024, 768, 12, 1, 1.0, s)]",
    "linear, 64-row panels": "[L.et_tile_plan_run(plan(768, 3072, 0.8), x, x, 4096, 1, s)]",
    "linear, chunks": "[L.et_tile_plan_run(plan(3072, 768, 0.8), x, x, m, 0, s) for m in (100, 3300, 16384)]",
    "linear + LayerNorm": "[L.et_tile_plan_run_ln(plan(k, 768, 0.8), x, x, x, x, x, 8192, s) for k in (768, 3072)]",
    "raw linear": "[L.et_tile_spmm_add_bias(x, x, x, x, x, m, 768, k, x, s) for m, k in ((64, 768), (4096, 768), (64, 3072))]",
    "dense product": "[L.et_row_spmm_add_bias(x, x, x, x, m, 768, 3072, s) for m in (2000, 8192, 65536)]",
    "projections and attention": "[L.et_qkv_attention(x, x, *[plan(768, 768, 0.8) for _ in range(3)], m, None, None, 128, 128, 768,"
                                 " 12, 4, 1.0, s) for m in (None, x)]",
    "layer tail": "[L.et_tile_plan_run_tail(plan(768, 768, 0.8), plan(768, 3072, 0.8), plan(3072, 768, 0.8), *[x] * 9, 8192, s)]",
    "layer tail in pairs": "[L.et_tile_plan_run_tail_ws(plan(768, 768, 0.8), plan(768, 3072, 0.8), plan(3072, 768, 0.8), *[x] * 9,"
                           " 2048, y, 1 << 27, s) for v in (1, 2, 3) if not L.et_tuning_set(b'tile_tail_pair', v)]",
    "layer": "[L.et_layer_flow_run(flow(37), x, x, x, x, x, x, m, None, None, x, x, x, x, 1.0, s) for m in (None, x)]",
    "compact linear + LayerNorm": "[L.et_tile_plan_run_scatter_ln(plan(k, 384, 0.0), x, x, y, x, 384, x, x, x, 768, 8192, s)"
                                  " for k in (768, 1024)]",
    "LayerNorm": "[L.et_skip_layernorm(x, x, x, x, 1000, 768, s)]",
}


@pytest.mark.parametrize("op", OTHER_STREAM)
def test_launches_take_the_device_of_their_stream(runtime, op):
    """a stream of the second device while the first one is current: functions, and the opt-in to large LDS, of the second
    device, whichever of the two was used first; the current device stays"""
    run(runtime, f"""
d = C.c_int()
for device in (1, 0, 1):
    s = stream(device)
    rt.two_devices_clear()
    for rc in {OTHER_STREAM[op]}:
        check(rc)
    ls = launches()
    assert ls and all(l[0] == device for l in ls), ls
    rt.hipGetDevice(C.byref(d))
    assert d.value == 0
""")


def test_static_scratch_is_that_of_the_streams_device(runtime):
    """et_OTF_attention_noalloc: every device has its own copy of the mask summary's array"""
    run(runtime, """
rt.two_devices_third(4)  # (the summary kernel: a word for 200 keys; mask, rows, summary, words)
for device in (1, 0):
    rt.two_devices_clear()
    check(L.et_OTF_attention_noalloc(x, x, x, x, x, 200, 768, 12, 1, None, 1.0, stream(device)))
    assert [l[0] for l in launches()] == [device, device]
    assert rt.two_devices_variable_of(0) == device
""")


def test_a_refused_opt_in_is_reported_and_nothing_launched(runtime):
    run(runtime, """
rt.two_devices_refuse(1)
for s in (None, stream(1)):
    assert L.et_OTF_attention(x, x, x, x, None, 1024, 768, 12, 1, None, 1.0, s) == -4
    assert L.et_tile_plan_run(plan(768, 3072, 0.8), x, x, 4096, 1, s) == -4
assert launches() == []
rt.two_devices_refuse(0)
check(L.et_OTF_attention(x, x, x, x, None, 1024, 768, 12, 1, None, 1.0, None))
""")


def test_a_tuning_key_holds_from_its_return_on_other_threads_too(runtime):
    """choices are kept per thread under the number of et_tuning_set calls: a launch that is being weighed while a key is
    set must not keep the old value's choice under the new number"""
    run(runtime, """
rows, values, threads = 4096, (C.c_int * 2)(0, 2), (C.c_uint * 2)()
p = plan(768, 3072, 0.8)
for i in range(2):
    check(L.et_tuning_set(b"tile_bm64", values[i]))  # 32-row panels, 64-row panels
    check(L.et_tile_plan_run(p, x, x, rows, 1, None))
    threads[i] = launches()[-1][1]
assert threads[0] != threads[1]
as_pointer = lambda f: C.cast(f, C.c_void_p)
assert rt.two_devices_race(as_pointer(L.et_tuning_set), as_pointer(L.et_tile_plan_run), p, x, rows, b"tile_bm64", values, threads,
                           20000) == 0
""")
