"""What the linears' host code launches, without a GPU: the library runs on a stand-in for the HIP runtime
(fakehip/fakehip.cpp), in which memory is host memory, a launch is only recorded and the test chooses what fails. Each
case runs in a child process."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "bitllm.c_amd", "libbitllm_hip.so")

SETUP = textwrap.dedent("""
    import ctypes as C, os, sys
    sys.path.insert(0, sys.argv[3])
    import numpy as np
    fake = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)
    import bitllm_hip as bh
    lib = bh.load()
    for n in ("fake_launch_arg1", "fake_launch_stream"):
        getattr(fake, n).restype = C.c_void_p
    vp = C.c_void_p

    def weight(N, K, g=128):
        codes, s = np.zeros((N, K // 4), np.uint8), np.ones((N, -(-K // g)) if g else N, np.float32)
        return bh.QWeight(bh.W_TERNARY, N, K, g, codes, s)

    _buf = np.zeros(1 << 18, np.uint8)
    X = vp((_buf.ctypes.data + 255) & ~255)   # rows that nothing reads or writes

    def spec(K, block=128):
        sp = bh.PrepSpec()
        sp.x, sp.ldx, sp.pre, sp.eps, sp.wht_block, sp.wht_norm = X, K, 1, 1e-5, block, 0.088
        return sp

    def linear(w, N, K, M, st=None):
        fake.fake_reset()
        return lib.eif_hip_qlinear_prep(w.h, C.byref(spec(K)), None, X, N, M, st)

    def glu(w, N, K, M, st=None):
        fake.fake_reset()
        return lib.eif_hip_qlinear_prep_glu(w.h, C.byref(spec(K)), X, N // 2, M, st)

    LIMIT, DEVICE = -4, -2
""")


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fakehip") / "libfakehip.so")
    src = os.path.join(ROOT, "tests", "fakehip", "fakehip.cpp")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", src, "-o", so], check=True)
    return so


def run(fake, body):
    r = subprocess.run([sys.executable, "-c", SETUP + textwrap.dedent(body), LIB, fake, os.path.join(ROOT, "bitllm.c_amd")],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_gated_call_reports_a_failed_prep_launch(fake):
    """A prep launch that the device refuses is the call's error: the gated form does not go on to its fused launch."""
    run(fake, """
        N, K = 512, 2560
        w = weight(N, K)
        assert glu(w, N, K, 4) == 0 and fake.fake_launches() == 2
        fake.fake_reset()
        fake.fake_fail_launch(0)
        assert lib.eif_hip_qlinear_prep_glu(w.h, C.byref(spec(K)), X, N // 2, 4, None) == DEVICE
        assert fake.fake_launches() == 1
    """)
