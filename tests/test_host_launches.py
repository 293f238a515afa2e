"""What the host code launches, without a device: the library runs in a child
process on stand-ins for the HIP calls (tests/c/fake_hip.c) that log them.
A launch that fails ends its call: the kernels after it would work on what it
should have written.  A call that is recorded into a graph after the same call
ran eagerly allocates, frees and waits for nothing: that would end the capture."""
import json
import os
import subprocess
import sys

import pytest

from conftest import ROOT

CHILD = r"""
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
fake.fake_reset.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_size_t]
sys.path.insert(0, sys.argv[2])
import ncmhip
lib = ncmhip.load()
lib.ncm_hip_set_error_mode(1)   # errors are returned, not fatal
assert lib.ncm_hip_init(0) == 0
P = [ctypes.c_void_p(0x10000000 * (i + 1)) for i in range(16)]   # operands: 16-byte aligned addresses, never read

def linear_fwd(M, N, K, off=0):
    lib.linear_fwd(ctypes.c_void_p(P[0].value + off), P[1], P[2], P[3], M, N, K)

def linear_bwd(M, N, K, off=0):
    lib.linear_bwd(ctypes.c_void_p(P[0].value + off), P[1], P[2], P[3], P[4], P[5], M, N, K)

def gated(M, N, K):
    lib.linear_fwd_gated(P[0], P[1], P[2], P[3], P[4], P[5], M, N, K, 1)

def vq(rows, V, D):
    lib.vq_argmin(P[0], P[1], P[2], rows, V, D)

def multiscale(rows, V, D, n):
    E, vocabs = (ctypes.c_void_p * n)(*[p.value for p in P[4:4 + n]]), (ctypes.c_int * n)(*[V] * n)
    lib.vq_quantize_multiscale(P[0], E, vocabs, n, 1, rows, D, P[1], P[2], P[3])

def call(name, args, fail=0, capture=0, limit=0):
    fake.fake_reset(fail, capture, limit)
    globals()[name](*args)
    err = lib.ncm_hip_last_error(None, 0)
    return {"error": err, "log": fake.fake_log().decode().split()}

print(json.dumps([call(*step) for step in json.loads(sys.argv[3])]))
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """host(steps): (name, args, fail, capture, limit) each, run in one process; their errors and logs."""
    fake = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "c", "fake_hip.c"), "-o", fake], check=True)

    def run(steps):
        out = subprocess.run([sys.executable, "-c", CHILD, fake, os.path.join(ROOT, "saphira-cncm_amd"),
                              json.dumps(steps)], check=True, capture_output=True, text=True, timeout=300)
        return json.loads(out.stdout)
    return run


def launches(result):
    return [w for w in result["log"] if not w.startswith("hip")]


CALLS = [("vq", (1000, 4096, 64)), ("vq", (1000, 100, 16)), ("multiscale", (1000, 4096, 64, 3)),
         ("multiscale", (1000, 60, 30, 2)), ("linear_fwd", (4096, 1024, 768)), ("linear_fwd", (512, 4864, 896)),
         ("linear_bwd", (4096, 3072, 768)), ("linear_bwd", (1000, 515, 1001)), ("linear_bwd", (64, 768, 768)),
         ("gated", (2048, 4864, 896))]


@pytest.mark.parametrize("name,args", CALLS)
def test_nothing_is_launched_after_a_failed_launch(host, name, args):
    whole = launches(host([(name, args)])[0])
    assert whole
    steps = [(name, args, 0)] + [(name, args, n) for n in range(1, len(whole) + 1)]
    for n, r in enumerate(host(steps)):
        assert (r["error"] != 0) == (n > 0)
        assert launches(r) == (whole[:n] if n else whole)


@pytest.mark.parametrize("name,args", CALLS + [("linear_fwd", (2048, 1152, 896)), ("linear_bwd", (4096, 768, 2304)),
                                               ("linear_bwd", (4096, 771, 2301)), ("linear_bwd", (4096, 768, 2304, 4))])
def test_capture_after_an_eager_call(host, name, args):
    eager, captured = host([(name, args), (name, args, 0, 1)])
    assert not eager["error"] and not captured["error"] and launches(captured)
    assert not {"hipMalloc", "hipFree", "hipStreamSynchronize"} & set(captured["log"])
    assert not any(w.startswith(("split_", "vq_screen16", "vq_pack")) for w in captured["log"])


def test_a_refused_workspace_leaves_the_smaller_one(host):
    """Where the device has no room for a call's packed operands the call runs on
    the FP32 kernels; calls that fit the workspace already held keep it, without
    allocating, freeing or waiting."""
    small, big = ("linear_fwd", (4096, 1024, 768)), ("linear_fwd", (16384, 3072, 768))
    first, refused, again, grown = host([small, (*big, 0, 0, 24 << 20), small, big])
    assert any(w.startswith("split_") for w in launches(first))
    assert not refused["error"] and all(w.startswith("gemm_") for w in launches(refused))
    assert not {"hipFree", "hipStreamSynchronize"} & set(refused["log"])
    assert not {"hipMalloc", "hipFree", "hipStreamSynchronize"} & set(again["log"])
    assert launches(again) == launches(first)
    assert any(w.startswith("split_") for w in launches(grown))
