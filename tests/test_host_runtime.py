"""The engine's host side on a HIP runtime of host memory (cpp/host_hip.cpp): kernels do nothing, so results mean nothing;
what is checked is which device is current, what is allocated, launched and replayed, and what a call leaves behind.

Each case runs in a process of its own (the runtime replaces HIP for the whole process): ``python test_host_runtime.py CASE``.
"""
import ctypes
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "cpp", "_build", "libhost_hip.so")


def _llama(**kw):
    from simplellminference_amd.model import LlamaModel, preset
    return LlamaModel(config=preset(kw.pop("preset", "tiny-gqa"), **kw.pop("over", {})), seed=1, **kw).init()


def _prompts(m, n):
    return [[(7 * b + i) % m.config.vocab_size for i in range(n)] for b in range(m.batch)]


# ---------------------------------------------------------------- cases (in the child)
def device_of_predict(H):
    """predict and predict_batch of a model on device 1 from a thread whose device is 0: what they allocate is on device 1,
    what they launch is launched there, and the thread's device is what it was."""
    for kw in (dict(w_dtype="f32", kv_dtype="f32"), dict(w_dtype="f16", batch=2)):
        m = _llama(device=1, **kw)
        H.hipSetDevice(0)
        before = H.hh_mallocs_on(0), H.hh_attributes_on(0), H.hh_mallocs_on(1)
        m.predict_batch(_prompts(m, 20), 24)
        assert H.hh_mallocs_on(1) > before[2], "the call allocates its scratch"
        assert (H.hh_mallocs_on(0), H.hh_attributes_on(0)) == before[:2], "memory or attributes of the other device"
        d = ctypes.c_int(-1)
        H.hipGetDevice(ctypes.byref(d))
        assert d.value == 0, "the caller's device"
        H.hipSetDevice(0)
        m.set_state_seq(0, 1, 0)
        m.step()
        m.close()
    assert H.hh_wrong_device() == 0, "launches on a stream of another device"


# ---------------------------------------------------------------- the tests
CASES = ["device_of_predict"]


@pytest.fixture(scope="module")
def host_hip():
    from simplellminference_amd import build
    build.ensure()
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    src = os.path.join(HERE, "cpp", "host_hip.cpp")
    part = f"{LIB}.{os.getpid()}"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", src, "-o", part], check=True)
    os.replace(part, LIB)
    return LIB


@pytest.mark.parametrize("case", CASES)
def test_host(host_hip, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    H = ctypes.CDLL(LIB, mode=ctypes.RTLD_GLOBAL)  # before libsli.so: its references to HIP end here
    H.hh_fail_size.argtypes = [ctypes.c_size_t]
    globals()[sys.argv[1]](H)
    print("ok", sys.argv[1])
