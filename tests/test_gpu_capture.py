"""Launches recorded between lancius_hip_capture_begin and _end, replayed with
other work of the same context between the replays: the graph keeps the scratch
memory it recorded, whatever the context needs afterwards, and a call that
needs scratch memory which a recording context does not have gets a kernel
without."""
import ctypes as C

import numpy as np
import pytest

import oracle
from lancius_amd import ACT_NONE, ACT_RELU, Device, prng
from tests.conftest import case

pytestmark = pytest.mark.gpu


class _Recorded:
    """The calls of `enqueue` as a graph on context d."""

    def __init__(self, d, enqueue):
        assert d.lib.lancius_hip_capture_begin(d.ctx) == 0, d.lib.lancius_hip_last_error()
        try:
            enqueue()
        finally:
            self.graph = C.c_void_p()
            rc = d.lib.lancius_hip_capture_end(d.ctx, C.byref(self.graph))
        assert rc == 0, d.lib.lancius_hip_last_error()
        self.lib = d.lib

    def replay(self, d):
        assert self.lib.lancius_hip_graph_launch(self.graph, d.ctx) == 0, self.lib.lancius_hip_last_error()
        d.synchronize()

    def destroy(self):
        self.lib.lancius_hip_graph_destroy(self.graph)


def _bits(a):
    return a.view(np.uint32)


def test_graph_keeps_its_scratch_memory():
    """A graph that uses the workspace (re-laid filters, split sums) and the
    arrival counters, replayed after the context has outgrown both and after
    it is gone.  What the context gave up would be handed out again: buffers
    filled in between must not reach the replays."""
    d, other = Device(0, own_stream=True), Device(0, own_stream=True)
    N, Ci, H, W, Co = 2, 24, 31, 29, 40
    Ho, Wo = (H + 2 - 3) // 2 + 1, (W + 2 - 3) // 2 + 1
    dy, w = prng.normal(1, (N, Co, Ho, Wo)), prng.normal(2, (Co, Ci, 3, 3), 0, 0.1)
    x, B, bias = prng.normal(3, (8, 2048)), prng.normal(4, (2048, 192)), prng.normal(5, (192,))
    g_dy, g_w, g_x, g_B, g_b = (d.upload(a) for a in (dy, w, x, B, bias))
    o_dx, o_y = d.alloc(4 * N * Ci * H * W), d.alloc(4 * 8 * 192)

    def enqueue():
        d.conv2d_bwd_input(o_dx, g_dy, g_w, N, Ci, H, W, Co, Ho, Wo, 3, 3, 2, 1)
        d.gemm(o_y, g_x, g_B, 8, 2048, 192, bias=g_b, act=ACT_RELU)

    def results():
        return d.download(o_dx, (N, Ci, H, W)), d.download(o_y, (8, 192))

    enqueue()
    want = results()
    y = oracle.relu(oracle.matmul(x, B) + bias.astype(np.float64)[None, :])
    assert oracle.normwise_error(want[1], y) <= oracle.tolerance(2048)
    case("graph recorded before its context outgrows its scratch memory")
    rec = _Recorded(d, enqueue)
    fills = []
    for rep, (m, k, n) in enumerate([(32, 4096, 4096), (32, 8192, 8192), (16, 2048, 300000)]):
        # slices of K: more partial sums, and more columns of counters, each time
        A_, B_, C_ = d.alloc(4 * m * k), d.alloc(4 * k * n), d.alloc(4 * m * n)
        d.fill(A_, 1.0, m * k)
        d.fill(B_, 1.0, k * n)
        d.gemm(C_, A_, B_, m, k, n)
        assert (d.download(C_, (m, n)) == float(k)).all()
        for b in (A_, B_, C_):
            b.free()
        fills += [other.alloc(1 << 20) for _ in range(8)]
        for b in fills:
            other.fill(b, 9.0, 1 << 18)
        other.synchronize()
        d.fill(o_dx, float("nan"), N * Ci * H * W)
        d.fill(o_y, float("nan"), 8 * 192)
        rec.replay(d)
        for got, ref in zip(results(), want):
            assert np.array_equal(_bits(got), _bits(ref)), rep
        for b in fills:
            assert (other.download(b, (1 << 18,)) == 9.0).all(), rep
    # the buffers are the context's to free, its memory goes with it
    host = [np.ascontiguousarray(a) for a in want]
    for b in fills:
        b.free()
    rec.destroy()
    for b in (g_dy, g_w, g_x, g_B, g_b, o_dx, o_y):
        b.free()
    d.close()
    other.close()
    assert all(np.isfinite(a).all() for a in host)


def test_graph_outlives_its_context():
    """Recorded on a context that is destroyed before the replays, which run on another."""
    d, other = Device(0, own_stream=True), Device(0, own_stream=True)
    A, B = prng.normal(11, (16, 4096)), prng.normal(12, (4096, 512))
    gA, gB, gC = other.upload(A), other.upload(B), other.alloc(4 * 16 * 512)
    d.gemm(gC, gA, gB, 16, 4096, 512)
    d.synchronize()
    want = other.download(gC, (16, 512))
    assert oracle.normwise_error(want, oracle.matmul(A, B)) <= oracle.tolerance(4096)
    case("graph whose context is gone")
    rec = _Recorded(d, lambda: d.gemm(gC, gA, gB, 16, 4096, 512))
    d.close()
    for rep in range(3):
        other.fill(gC, float("nan"), 16 * 512)
        fill = other.alloc(4 << 20)
        other.fill(fill, 9.0, 1 << 20)
        rec.replay(other)
        assert np.array_equal(_bits(other.download(gC, (16, 512))), _bits(want)), rep
        assert (other.download(fill, (1 << 20,)) == 9.0).all(), rep
        fill.free()
    rec.destroy()
    for b in (gA, gB, gC):
        b.free()
    other.close()


def _gemm_split_k(d):
    M, K, N = 768, 4096, 1024
    A, B = prng.normal(21, (M, K)), prng.normal(22, (K, N))
    gA, gB, o = d.upload(A), d.upload(B), d.alloc(4 * M * N)
    return lambda: d.gemm(o, gA, gB, M, K, N), o, (M, N), oracle.matmul(A, B), K


def _conv_ragged(d):
    N, Ci, H, W, Co = 1, 13, 64, 64, 51
    x, w = prng.normal(23, (N, Ci, H, W)), prng.normal(24, (Co, Ci, 5, 5), 0, 0.06)
    gx, gw, o = d.upload(x), d.upload(w), d.alloc(4 * N * Co * H * W)
    return (lambda: d.conv2d(o, gx, gw, None, N, Ci, H, W, Co, 5, 5, 1, 2, ACT_NONE), o, (N, Co, H, W),
            oracle.conv2d(x, w, 1, 2, False), Ci * 25)


def _conv_gradient_strided(d):
    N, Ci, H, W, Co = 2, 24, 31, 29, 40
    Ho, Wo = (H + 2 - 3) // 2 + 1, (W + 2 - 3) // 2 + 1
    dy, w = prng.normal(25, (N, Co, Ho, Wo)), prng.normal(26, (Co, Ci, 3, 3), 0, 0.1)
    gd, gw, o = d.upload(dy), d.upload(w), d.alloc(4 * N * Ci * H * W)
    return (lambda: d.conv2d_bwd_input(o, gd, gw, N, Ci, H, W, Co, Ho, Wo, 3, 3, 2, 1), o, (N, Ci, H, W),
            oracle.conv2d_bwd_input(dy, w, (N, Ci, H, W), 2, 1), Co * 9)


def _loss(d):
    rows, cols = 1000, 37
    x, y = prng.normal(27, (rows, cols)), np.zeros((rows, cols), np.float32)
    y[np.arange(rows), np.arange(rows) % cols] = 1.0
    gx, gy, o = d.upload(x), d.upload(y), d.alloc(4)
    x64 = x.astype(np.float64)
    lse = np.log(np.exp(x64 - x64.max(1, keepdims=True)).sum(1)) + x64.max(1)
    return (lambda: d.cross_entropy(o, gx, gy, rows, cols), o, (1,),
            np.asarray([np.mean(lse - x64[np.arange(rows), np.arange(rows) % cols])]), cols)


@pytest.mark.parametrize("call", [_gemm_split_k, _conv_ragged, _conv_gradient_strided, _loss],
                         ids=["gemm split K", "conv ragged", "conv gradient stride 2", "loss"])
def test_capture_without_scratch_memory(call):
    """Each recorded first on a context without scratch memory (a kernel that
    needs none), then on the same context after the call has run (the kernel
    that it has outside a capture, hence its bits)."""
    d = Device(0, own_stream=True)
    enqueue, out, shape, ref, K = call(d)
    n = int(np.prod(shape))
    case(f"recorded on a fresh context: {call.__name__}")
    fresh = _Recorded(d, enqueue)
    enqueue()
    eager = d.download(out, shape)
    assert oracle.normwise_error(eager, ref) <= oracle.tolerance(K)
    ready = _Recorded(d, enqueue)
    first = None
    for rep in range(3):
        for rec in (fresh, ready):
            d.fill(out, float("nan"), n)
            rec.replay(d)
            got = d.download(out, shape)
            if rec is ready:
                assert np.array_equal(_bits(got), _bits(eager)), rep
            else:
                assert oracle.normwise_error(got, ref) <= oracle.tolerance(K), rep
                first = got if first is None else first
                assert np.array_equal(_bits(got), _bits(first)), rep
        enqueue()
        d.synchronize()
    fresh.destroy()
    ready.destroy()
    d.close()
