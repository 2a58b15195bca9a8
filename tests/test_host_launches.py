"""What the linears' host code launches, without a GPU: the library runs on a stand-in for the HIP runtime
(fakehip/fakehip.cpp), in which memory is host memory, a launch is only recorded and the test chooses what fails. Each
case runs in a child process."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT
from test_gpu_qlinear import TILE_SPLIT

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


ROWS_CALLS = """
    fake.fake_read_arg1(1)
    N, K = 512, 4096
    w = weight(N, K)

    def rows(call, M, st=None):
        assert call(w, N, K, M, st) == 0
        return fake.fake_launches(), fake.fake_launch_arg1(0)
"""


def test_rows_calls_in_a_capture_are_one_launch(fake):
    """3 to 8 rows: a prep launch and the GEMV outside a capture; inside one the single launch, also on a stream that
    has a rows buffer, and nothing is allocated."""
    run(fake, ROWS_CALLS + """
    for call in (linear, glu):
        for M in (3, 8):
            for st in (None, 0x100):
                assert rows(call, M, st)[0] == 2
                n = fake.fake_mallocs()
                fake.fake_capturing(1)
                assert rows(call, M, st)[0] == 1 and rows(call, M, 0x200)[0] == 1 and fake.fake_mallocs() == n
                fake.fake_capturing(0)
    """)


def test_rows_buffers(fake):
    """One rows buffer a device and stream, which stays where it is; none for the handle that means a stream per thread;
    64 at most; all given back with the last resident weight."""
    run(fake, ROWS_CALLS + """
    w2 = weight(256, 6144)
    live = fake.fake_live()
    _, p = rows(linear, 3)
    assert fake.fake_live() == live + 1
    assert linear(w2, 256, 6144, 8) == 0 and fake.fake_launches() == 2 and fake.fake_launch_arg1(0) == p
    assert rows(glu, 5)[1] == p and rows(linear, 8, 0x100)[1] != p and fake.fake_live() == live + 2
    fake.fake_device(1)
    assert rows(linear, 4)[1] not in (p, None) and fake.fake_live() == live + 3
    fake.fake_device(0)
    assert rows(linear, 4) == (2, p)
    assert rows(linear, 4, 2)[0] == 1   # hipStreamPerThread
    for st in range(0x200, 0x200 + 100):
        assert rows(linear, 4, st)[0] in (1, 2)
    assert fake.fake_live() == live + 64 and rows(linear, 4)[0] == 2 and rows(linear, 4, 0x300)[0] == 1
    w2.close()
    assert rows(linear, 4) == (2, p)
    w.close()
    assert fake.fake_live() == 0
    w = weight(N, K)
    assert rows(linear, 4, 0x300)[0] == 2
    """)


def test_rows_call_without_memory(fake):
    """Where the rows buffer cannot be allocated the call is the single launch, as for one row, and reports no error."""
    run(fake, ROWS_CALLS + """
    for call in (linear, glu):
        fake.fake_reset()
        fake.fake_fail_malloc(1)
        f = lib.eif_hip_qlinear_prep_glu if call is glu else lib.eif_hip_qlinear_prep
        a = (w.h, C.byref(spec(K))) + (() if call is glu else (None,))
        assert f(*a, X, N, 4, None) == 0 and fake.fake_launches() == 1
    """)


@pytest.mark.parametrize("fmt,N,K,block,pre,first", [
    # the first row count of two launches; 9: none
    (1, 2560, 512, 0, 1, 8), (1, 2560, 512, 128, 1, 6), (2, 640, 640, 0, 1, 8),
    (2, 2560, 1024, 0, 1, 7), (1, 6912, 1024, 0, 1, 6), (1, 6912, 1024, 128, 1, 5), (3, 7168, 1024, 0, 1, 6),
    (2, 2560, 1536, 0, 1, 6), (1, 6912, 1536, 0, 1, 4), (1, 2560, 1536, 128, 1, 5), (1, 4096, 1152, 128, 1, 5),
    (2, 2560, 2560, 0, 1, 4), (1, 2560, 2560, 0, 1, 5), (1, 2560, 2560, 128, 1, 4), (1, 13824, 2560, 128, 1, 3),
    (1, 2560, 4096, 0, 1, 4), (2, 2560, 4096, 0, 1, 3), (1, 2560, 6912, 128, 1, 3), (3, 65536, 1024, 0, 1, 3),
    (1, 2560, 1024, 0, 0, 9), (2, 6912, 1024, 0, 0, 8), (1, 2560, 2048, 128, 0, 7), (2, 2560, 2560, 0, 0, 6),
    (1, 6912, 2560, 128, 0, 4), (1, 2560, 4864, 0, 0, 5), (3, 65536, 1024, 0, 0, 3),
])
def test_rows_where_two_launches_pay(fake, fmt, N, K, block, pre, first):
    """Rows are prepped in a launch of their own only where that is faster than the fused form, which is a matter of the
    row's columns, norm and rotation and of the matrix's rows."""
    run(fake, f"""
    fmt, N, K, block, first = {fmt}, {N}, {K}, {block}, {first}
    g = 128 if block else 0
    if fmt == 1:
        w = weight(N, K, g)
    else:
        w = bh.QWeight(fmt, N, K, 0, np.zeros((N, K if fmt == 2 else K // 2), np.int8), np.ones(N, np.float32))
    sp = spec(K, block)
    sp.pre = {pre}
    for M in range(2, 9):
        fake.fake_reset()
        assert lib.eif_hip_qlinear_prep(w.h, C.byref(sp), None, X, N, M, None) == 0
        assert fake.fake_launches() == (2 if M >= first else 1), M
    """)


@pytest.mark.parametrize("M,K,ldq,pre,block,wave_a_row", [
    (1023, 2560, 2560, 1, 128, False), (1024, 2560, 2560, 1, 128, True), (3001, 2304, 2304, 1, 128, False),
    (1024, 2336, 2336, 1, 32, True), (3001, 2688, 2688, 1, 128, False), (3001, 2560, 2560, 1, 512, False),
    (3001, 2560, 2560, 0, 128, False), (3001, 2560, 2560, 2, 128, False),
    (1023, 896, 1024, 1, 0, False), (1024, 896, 1024, 1, 0, True), (2047, 2880, 3072, 1, 0, False),
    (2048, 2880, 3072, 1, 0, True), (3001, 4096, 4096, 1, 0, True), (3001, 4224, 4352, 1, 0, False),
    (3001, 896, 1024, 0, 0, False),
])
def test_prep_of_a_batch(fake, M, K, ldq, pre, block, wave_a_row):
    """A batch's prep gives a row a wave (workgroups of four rows) only where that is faster than a workgroup a row."""
    run(fake, f"""
    M, K, ldq, pre, block = {M}, {K}, {ldq}, {pre}, {block}
    sp = spec(K, block)
    sp.pre, sp.x2 = pre, X
    fake.fake_reset()
    assert lib.eif_hip_prep_spec_rows(C.byref(sp), K, X, ldq, X, M, None) == 0
    assert fake.fake_launches() == 1
    assert (fake.fake_launch_grid(0), fake.fake_launch_block(0) == 256) == \\
        ((-(-M // 4), True) if {wave_a_row} else (M, fake.fake_launch_block(0) == 256))
    """)


@pytest.mark.parametrize("N,K,g,M,tm,tn,ks", TILE_SPLIT)
def test_split_shapes_take_the_tiled_form(fake, N, K, g, M, tm, tn, ks):
    """The shapes of test_gemm_tile_split run the register-tiled GEMM, with that tile and that many splits."""
    run(fake, f"""
    N, K, g, M, tm, tn, ks = {N}, {K}, {g}, {M}, {tm}, {tn}, {ks}
    w = weight(N, K, g)
    fake.fake_reset()
    assert lib.eif_hip_qlinear_ex(w.h, X, w.kpad, X, None, X, N, M, bh.PATH_GEMM, None) == 0
    tiles = -(-M // tm) * -(-(-(-N // 64) * 64) // tn)
    assert fake.fake_launches() == 1
    assert (fake.fake_launch_grid(0), fake.fake_launch_block(0)) == (tiles * ks, 2 * tn)
    """)
