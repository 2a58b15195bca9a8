"""The hot path captured into a HIP graph: every replay, with eager work and synchronisations in between,
matches the eager result bit for bit (the path records no memset nodes)."""
import ctypes as C

import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


def test_graph_replays_match_eager(gpu):
    import torch
    dev = torch.device("cuda:0")
    N, K, g, M = 6912, 2560, 128, 1
    w, s = synth.ternary_weight((60,), N, K, g)
    qw = gpu.QWeight(gpu.W_TERNARY, N, K, g, w, s)
    x = torch.from_numpy(synth.activations((61,), M, K)).to(dev)
    xq = torch.zeros((M, qw.kpad), dtype=torch.int8, device=dev)
    xs = torch.zeros(M, dtype=torch.float32, device=dev)
    y = torch.zeros((M, N), dtype=torch.float32, device=dev)
    norm = gpu.wht_norm(128)

    def step():
        gpu.prep_rows(x, xq, xs, 128, norm)
        qw.linear(xq, xs, y, path=gpu.PATH_GEMV)

    step()
    torch.cuda.synchronize()
    want = y.cpu().numpy().copy()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for r in range(4):
        y.fill_(float("nan"))
        xq.fill_(3)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"replay {r} differs"
        # eager work between replays
        step()
        torch.cuda.synchronize()
    qw.close()


ROWS = [
    # fmt, N, K, group, M, WHT block: calls of 3 to 8 rows, two launches eagerly and one in a capture
    ("tern", 3840, 2560, 128, 4, 128),
    ("tern", 2560, 6912, 96, 8, 128),
    ("tern", 100, 640, 64, 6, 64),
    ("tern", 512, 2560, 0, 5, 0),
    ("int8", 896, 4864, 0, 3, 0),
    ("int8", 1000, 896, 0, 7, 0),
    ("int4", 3584, 1024, 0, 8, 0),
    ("glu", 13824, 2560, 128, 3, 128),
    ("glu", 13824, 2560, 128, 8, 128),
    ("glu", 512, 640, 128, 8, 0),
]


class RowsCall:
    """One eif_hip_qlinear_prep (or _glu) call of M rows, with rows of its own."""

    def __init__(self, gpu, qw, fmt, M, block, seed):
        import torch
        dev = torch.device("cuda:0")
        self.gpu, self.qw, self.fmt, self.M = gpu, qw, fmt, M
        self.x = torch.from_numpy(synth.activations((62, seed), M, qw.cols)).to(dev)
        self.nw = torch.from_numpy((1.0 + 0.1 * synth.rng(63, seed).standard_normal(qw.cols)).astype(np.float32)).to(dev)
        self.spec = gpu.prep_spec(self.x, gpu.PRE_RMS, None, self.nw, 1e-5, None, block, gpu.wht_norm(block) if block else 1.0)
        self.y = torch.full((M, qw.rows // (2 if fmt == "glu" else 1)), float("nan"), dtype=torch.float32, device=dev)

    def __call__(self):
        lib, y = self.gpu.load(), self.y
        tail = (self.gpu.ptr(y), y.stride(0), self.M, self.gpu.stream_ptr())
        if self.fmt == "glu":
            rc = lib.eif_hip_qlinear_prep_glu(self.qw.h, C.byref(self.spec), *tail)
        else:
            rc = lib.eif_hip_qlinear_prep(self.qw.h, C.byref(self.spec), None, *tail)
        assert rc == 0, rc

    def bits(self):
        return self.y.cpu().numpy().view(np.uint32).copy()


def rows_weight(gpu, fmt, N, K, g):
    if fmt in ("tern", "glu"):
        return gpu.QWeight(gpu.W_TERNARY, N, K, g, *synth.ternary_weight((64, N, K, g), N, K, g))
    if fmt == "int8":
        return gpu.QWeight(gpu.W_INT8, N, K, 0, *synth.int8_weight((65, N, K), N, K))
    return gpu.QWeight(gpu.W_INT4, N, K, 0, *synth.int4_weight((66, N, K), N, K))


@pytest.mark.parametrize("fmt,N,K,g,M,block", ROWS)
def test_captured_rows(gpu, fmt, N, K, g, M, block):
    """Captured calls of 3 to 8 rows give the bits of eager ones at every replay, whether the capture stream had such calls
    before or not; and two graphs captured on one stream, replayed on two streams at once beside eager calls on the capture
    stream, keep to their own rows."""
    import torch
    qw = rows_weight(gpu, fmt, N, K, g)
    a, b, c = (RowsCall(gpu, qw, fmt, M, block, seed) for seed in (0, 1, 2))
    for call in (a, b, c):
        call()
    torch.cuda.synchronize()
    want = [call.bits() for call in (a, b, c)]
    used = torch.cuda.Stream()
    with torch.cuda.stream(used):
        c()   # `used` has its rows buffer
    torch.cuda.synchronize()
    graphs = []
    for call, st in ((a, torch.cuda.Stream()), (a, used), (b, used)):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            call()
        graphs.append(graph)
    for graph in graphs[:2]:
        for r in range(3):
            a.y.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(a.bits(), want[0]), r
            b()   # eager work between replays
            torch.cuda.synchronize()
            assert np.array_equal(b.bits(), want[1]), r
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    for call in (a, b, c):
        call.y.fill_(float("nan"))
    torch.cuda.synchronize()
    for _ in range(20):
        with torch.cuda.stream(s1):
            graphs[1].replay()
        with torch.cuda.stream(s2):
            graphs[2].replay()
        with torch.cuda.stream(used):
            c()
    torch.cuda.synchronize()
    assert [np.array_equal(call.bits(), w) for call, w in zip((a, b, c), want)] == [True] * 3
    qw.close()


def test_rows_buffer_during_a_capture(gpu):
    """A stream's first eager call of several rows, while another stream is being captured by the same thread, allocates
    its rows buffer without ending the capture."""
    import torch
    qw = rows_weight(gpu, "tern", 512, 4096, 128)
    a, b = (RowsCall(gpu, qw, "tern", 4, 128, seed) for seed in (3, 4))
    a()
    b()
    torch.cuda.synchronize()
    want = [a.bits(), b.bits()]
    a.y.fill_(float("nan"))
    b.y.fill_(float("nan"))
    torch.cuda.synchronize()
    st, fresh = torch.cuda.Stream(), C.c_void_p()
    hip = C.CDLL(next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln))
    assert hip.hipStreamCreateWithFlags(C.byref(fresh), 1) == 0   # not one that an earlier test used
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        a()
        with torch.cuda.stream(torch.cuda.ExternalStream(fresh.value)):
            b()
    torch.cuda.synchronize()
    assert np.array_equal(b.bits(), want[1])
    graph.replay()
    torch.cuda.synchronize()
    assert np.array_equal(a.bits(), want[0])
    qw.close()
    assert hip.hipStreamDestroy(fresh) == 0


def test_rows_calls_of_two_threads(gpu):
    """Two threads that issue calls of several rows on one stream share its rows buffer and keep to their own rows."""
    import threading

    import torch
    qw = rows_weight(gpu, "tern", 512, 4096, 128)
    calls = [RowsCall(gpu, qw, "tern", 8, 128, seed) for seed in (5, 6)]
    for call in calls:
        call()
    torch.cuda.synchronize()
    want = [call.bits() for call in calls]
    outs = [[torch.full_like(call.y, float("nan")) for _ in range(40)] for call in calls]
    failed = []

    def issue(call, ys):
        try:
            for y in ys:
                call.y = y
                call()
        except BaseException as e:   # an assertion in a thread is not the test's own
            failed.append(e)

    threads = [threading.Thread(target=issue, args=a) for a in zip(calls, outs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed
    for ys, w in zip(outs, want):
        assert all(np.array_equal(y.cpu().numpy().view(np.uint32), w) for y in ys)
    qw.close()
