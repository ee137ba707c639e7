"""The GEMM over packed bf16 operands (packed.hip, REHIP_GEMM_PACKED=2: at every shape it takes)
against an f64 product, at the edges of its tiles (64 .. 256), fragments (32 rows x 16 k), stages
(32 k) and K slices; the operands packed in pieces; its workspaces over streams and under capture.

Bounds per output, relative to sum |w x|: bf16 has 8 significant bits, so a rounding is off by at most
2^-8 and a bf16-mode product by 2^-7 + 2^-16; in f32 mode a remainder is at most 2^-8 of its value and
its rounding leaves 2^-16, so a product is off by 2^-16 for either operand and 2^-16 for the dropped
lo x lo (and 2^-32). The f32 sums add K roundings of 2^-24, whatever the MFMAs' order."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle as O
import rehip
from rehip import hip, synth

pytestmark = pytest.mark.gpu
B = hip.DeviceBuffer
TYPES = [rehip.Q4_0, rehip.Q5_0, rehip.Q8_0, rehip.Q4_K, rehip.Q5_K, rehip.Q6_K, rehip.F32, rehip.F16, rehip.BF16]
MODES = [rehip.MODE_BF16, rehip.MODE_F32]


def weights(rng, t, m, n):
    v = rng.standard_normal((m, n)).astype(np.float32)
    if t == rehip.F32:
        return v.view(np.uint8).reshape(-1)
    if t == rehip.F16:
        return v.astype(np.float16).view(np.uint8).reshape(-1)
    if t == rehip.BF16:
        return (v.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8).reshape(-1)
    return synth.weight_bytes(rng, t, m, n)


def product(t, w, m, n, x, rows):
    deq = O.dequant(t, w).reshape(m, -1)[:, :n].astype(np.float64)
    xx = x.reshape(rows, n).astype(np.float64)
    return xx @ deq.T, np.abs(xx) @ np.abs(deq).T


def check(got, want, n, mode):
    exact, absd = want
    rel = (2.0 ** -7 + 2.0 ** -16 if mode == rehip.MODE_BF16 else 3.01 * 2.0 ** -16) + n * 2.0 ** -24
    assert np.all(np.abs(got.reshape(exact.shape) - exact) <= rel * absd)


def run(q, dx, rows, m, mode, call="matmul_dev", stream=None):
    dy = B(rows * m * 4)
    getattr(q, call)(dx, rows, dy, mode, stream=stream)
    hip.synchronize()
    return dy.download(np.float32, rows * m)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("m,n,rows", [(1, 32, 65), (64, 64, 128), (70, 256, 100), (193, 96, 257), (129, 4864, 130),
                                      (257, 1056, 66), (600, 288, 300)])
def test_against_f64(t, mode, m, n, rows, monkeypatch):
    monkeypatch.setenv("REHIP_GEMM_PACKED", "2")
    rng = np.random.default_rng(1000 + t + m + rows)
    w, x = weights(rng, t, m, n), synth.activations(rng, rows, n)
    q = rehip.QMat.from_bytes(t, w, m, n)
    dx, want = B.from_array(x), product(t, w, m, n, x, rows)
    got = run(q, dx, rows, m, mode)
    check(got, want, n, mode)
    assert np.array_equal(run(q, dx, rows, m, mode), got)
    assert np.array_equal(run(q, dx, rows, m, mode, "matmul_noalloc_dev"), got)
    q.close()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("m,n,rows", [(4864, 896, 512), (1024, 512, 2100), (300, 2048, 400)])
def test_planned_tiles(mode, m, n, rows):
    """Shapes that the planner gives its larger tiles, in the default dispatch."""
    rng = np.random.default_rng(m + rows)
    w, x = weights(rng, rehip.Q5_K, m, n), synth.activations(rng, rows, n)
    q = rehip.QMat.from_bytes(rehip.Q5_K, w, m, n)
    check(run(q, B.from_array(x), rows, m, mode), product(rehip.Q5_K, w, m, n, x, rows), n, mode)
    q.close()


@pytest.mark.parametrize("t,m,n,rows,mode", [(rehip.Q4_K, 128, 8192, 512, rehip.MODE_BF16),
                                             (rehip.Q4_K, 128, 8192, 512, rehip.MODE_F32),
                                             (rehip.F16, 256, 2048, 256, rehip.MODE_BF16),
                                             (rehip.F32, 512, 4096, 384, rehip.MODE_F32)])
def test_small_products_are_not_packed(t, m, n, rows, mode):
    """Shapes where packing costs more than it gives run the unpacked GEMM: its bits (other K slices than the
    packed one's)."""
    rng = np.random.default_rng(m + rows)
    q = rehip.QMat.from_bytes(t, weights(rng, t, m, n), m, n)
    dx = B.from_array(synth.activations(rng, rows, n))
    got = {}
    for knob in ("0", "1", "2"):
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv("REHIP_GEMM_PACKED", knob)
            got[knob] = run(q, dx, rows, m, mode)
    assert np.array_equal(got["1"], got["0"]) and not np.array_equal(got["2"], got["0"])
    q.close()


@pytest.mark.parametrize("t", [rehip.F16, rehip.F32])
def test_dense_k_remainders(t, monkeypatch):
    """Dense rows need whole 8-element units only: K that ends inside a fragment and a stage."""
    monkeypatch.setenv("REHIP_GEMM_PACKED", "2")
    for n in (8, 24, 40, 200):
        rng = np.random.default_rng(n)
        w, x = weights(rng, t, 100, n), synth.activations(rng, 70, n)
        q = rehip.QMat.from_bytes(t, w, 100, n)
        for mode in MODES:
            check(run(q, B.from_array(x), 70, 100, mode), product(t, w, 100, n, x, 70), n, mode)
        q.close()


def test_bf16_weights_have_no_remainder():
    """BF16 weights in f32 mode are one plane: an infinite weight meets both parts of x (of one sign here) and
    stays infinite, as in the unpacked GEMM; the others' outputs are the unpacked GEMM's to 32-bit sums."""
    m, n, rows = 300, 512, 260
    rng = np.random.default_rng(13)
    w = rng.standard_normal((m, n)).astype(np.float32)
    w[5, 17], w[40, 0] = np.inf, -np.inf
    q = rehip.QMat.from_bytes(rehip.BF16, (w.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8).reshape(-1), m, n)
    x = rng.standard_normal((rows, n)).astype(np.float32)
    x[:, [0, 17]] = 1 + 2.0 ** -10
    got = []
    for knob in ("2", "0"):
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv("REHIP_GEMM_PACKED", knob)
            got.append(run(q, B.from_array(x), rows, m, rehip.MODE_F32).reshape(rows, m))
    assert np.all(got[0][:, 5] == np.inf) and np.all(got[0][:, 40] == -np.inf)
    assert np.array_equal(np.isfinite(got[0]), np.isfinite(got[1]))
    fine = np.isfinite(w).all(1)
    absd = np.abs(x).astype(np.float64) @ np.abs(w[fine]).astype(np.float64).T
    # two products per pair, so 2 n additions of 2^-24 in either order
    assert np.all(np.abs(got[0][:, fine] - got[1][:, fine]) <= 2 * 2 * n * 2.0 ** -24 * absd)
    q.close()


def test_operands_in_pieces():
    """Operands beyond the no-allocation scratch are packed and multiplied in pieces: the same bits."""
    t, m, n, rows = rehip.Q4_0, 700, 16384, 600
    rng = np.random.default_rng(5)
    q = rehip.QMat.from_bytes(t, weights(rng, t, m, n), m, n)
    dx = B.from_array(synth.activations(rng, rows, n))
    for mode in MODES:
        assert np.array_equal(run(q, dx, rows, m, mode), run(q, dx, rows, m, mode, "matmul_noalloc_dev"))
    q.close()


@pytest.mark.parametrize("t,m,n,rows,pieces", [(rehip.Q4_0, 28672, 1024, 1024, True), (rehip.F16, 4096, 4096, 512, True),
                                               (rehip.Q4_0, 4096, 4096, 512, False),
                                               (rehip.Q4_0, 2048, 8192, 1024, False),
                                               (rehip.F16, 2048, 8192, 1024, False)])
def test_pieces_only_where_they_fill_the_gpu(t, m, n, rows, pieces):
    """The no-allocation entry point with operands beyond its scratch: in pieces of the same bits, or the
    unpacked GEMM's bits where the pieces would be small or the rows few."""
    rng = np.random.default_rng(m)
    q = rehip.QMat.from_bytes(t, weights(rng, t, m, n), m, n)
    dx = B.from_array(synth.activations(rng, rows, n))
    got = run(q, dx, rows, m, rehip.MODE_F32, "matmul_noalloc_dev")
    with pytest.MonkeyPatch.context() as mp:
        if not pieces:
            mp.setenv("REHIP_GEMM_PACKED", "0")
        assert np.array_equal(run(q, dx, rows, m, rehip.MODE_F32), got)
    q.close()


def test_streams_and_capture():
    """More live streams than workspaces, two matrices in turn and no synchronisation in between; then a
    captured call (the tiled GEMM) replayed between eager ones."""
    m, n, rows = 640, 512, 400
    rng = np.random.default_rng(6)
    qs, dx, want = [], [], []
    for t in (rehip.Q6_K, rehip.Q8_0):
        w, x = weights(rng, t, m, n), synth.activations(rng, rows, n)
        qs.append(rehip.QMat.from_bytes(t, w, m, n))
        dx.append(B.from_array(x))
        want.append(product(t, w, m, n, x, rows))
    streams = [hip.Stream() for _ in range(10)]
    ys = [B(rows * m * 4) for _ in range(20)]
    for i in range(20):
        qs[i % 2].matmul_dev(dx[i % 2], rows, ys[i], rehip.MODE_F32, stream=streams[i // 2])
    hip.synchronize()
    for i in range(20):
        check(ys[i].download(np.float32, rows * m), want[i % 2], n, rehip.MODE_F32)
    y = B(rows * m * 4)
    g = hip.Graph(streams[0], lambda: qs[0].matmul_dev(dx[0], rows, y, rehip.MODE_F32, stream=streams[0]))
    for _ in range(3):
        g.launch()
        qs[1].matmul_dev(dx[1], rows, ys[1], rehip.MODE_F32, stream=streams[1])
        hip.synchronize()
        check(y.download(np.float32, rows * m), want[0], n, rehip.MODE_F32)
        check(ys[1].download(np.float32, rows * m), want[1], n, rehip.MODE_F32)
    g.destroy()
    for s in streams:
        s.destroy()
    for q in qs:
        q.close()


def test_streams_come_and_go():
    """Streams made, used and destroyed while their work may still run, more of them than workspaces, and
    new ones (which may get old handles) in their place: every call gets the bits of the first."""
    m, n, rows = 896, 4864, 400
    rng = np.random.default_rng(7)
    q = rehip.QMat.from_bytes(rehip.Q6_K, weights(rng, rehip.Q6_K, m, n), m, n)
    big = rehip.QMat.from_bytes(rehip.Q4_0, weights(rng, rehip.Q4_0, 4096, 4096), 4096, 4096)
    dx, dxb = B.from_array(synth.activations(rng, rows, n)), B.from_array(synth.activations(rng, rows, 4096))
    want, yb = run(q, dx, rows, m, rehip.MODE_F32), B(rows * 4096 * 4)
    for turn in range(4):
        streams = [hip.Stream() for _ in range(6 + turn)]
        ys = [B(rows * m * 4) for _ in streams]
        for s, y in zip(streams, ys):
            if turn == 2:
                big.matmul_dev(dxb, rows, yb, rehip.MODE_F32, stream=s)      # a larger workspace on the way
            q.matmul_dev(dx, rows, y, rehip.MODE_F32, stream=s)
        for s in streams:
            s.destroy()
        again = hip.Stream()
        y2 = B(rows * m * 4)
        q.matmul_dev(dx, rows, y2, rehip.MODE_F32, stream=again)
        hip.synchronize()
        for y in ys + [y2]:
            assert np.array_equal(y.download(np.float32, rows * m), want)
        again.destroy()
    q.close()
    big.close()


def test_threads():
    """More threads than workspaces, each with its own matrix and stream (two of them with the per-thread
    default stream, one handle for two streams): every call gets its own product."""
    m, n, rows = 640, 1024, 400
    rng = np.random.default_rng(10)
    jobs = []
    for i in range(6):
        q = rehip.QMat.from_bytes(rehip.Q8_0, weights(rng, rehip.Q8_0, m, n), m, n)
        x = B.from_array(synth.activations(rng, rows, n))
        jobs.append((q, x, run(q, x, rows, m, rehip.MODE_F32), [B(rows * m * 4) for _ in range(20)]))
    errors = []

    def work(i):
        try:
            q, x, _, ys = jobs[i]
            s = hip.Stream() if i < 4 else None
            for y in ys:                       # (hipStreamPerThread is the handle 2)
                q.matmul_dev(x, rows, y, rehip.MODE_F32, stream=s or 2)
            if s:
                s.destroy()
        except Exception as e:                 # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    hip.synchronize()
    assert not errors
    for q, _, want, ys in jobs:
        for y in ys:
            assert np.array_equal(y.download(np.float32, rows * m), want)
        q.close()


def test_results_reach_the_host():
    """The workspace's event carries no system-scope release: outputs still reach the host by a copy on the
    call's stream, by one on another stream after a synchronize, and written into pinned host memory."""
    m, n, rows = 896, 4864, 400
    rng = np.random.default_rng(9)
    q = rehip.QMat.from_bytes(rehip.Q6_K, weights(rng, rehip.Q6_K, m, n), m, n)
    dx = [B.from_array(synth.activations(rng, rows, n)) for _ in range(2)]
    want = [run(q, x, rows, m, rehip.MODE_BF16) for x in dx]
    H, y, size = hip.hip(), B(rows * m * 4), C.c_size_t(rows * m * 4)
    pinned, on_device = C.c_void_p(), C.c_void_p()
    hip.check(H.hipHostMalloc(C.byref(pinned), size, 0))
    hip.check(H.hipHostGetDevicePointer(C.byref(on_device), pinned, 0))
    got = np.ctypeslib.as_array(C.cast(pinned, C.POINTER(C.c_float)), (rows * m,))
    s, other = hip.Stream(), hip.Stream()
    for i in range(30):
        x, w = dx[i % 2], want[i % 2]
        for way in (s, other, None):
            got[:] = -1
            q.matmul_dev(x, rows, y if way else on_device.value, rehip.MODE_BF16, stream=s)
            if way is not s:
                s.synchronize()
            if way:
                hip.check(H.hipMemcpyAsync(pinned, C.c_void_p(y.ptr), size, 2, C.c_void_p(way.handle)))
                way.synchronize()
            assert np.array_equal(got, w), (i, way)
    del got
    hip.check(H.hipHostFree(pinned))
    for o in (s, other):
        o.destroy()
    q.close()


def test_capture_after_eager_call_keeps_its_slices():
    """A graph captured after an eager call (which ran on packed operands) takes the tiled GEMM with its
    K slices: the bits of a call that never packs."""
    m, n, rows = 896, 4864, 400
    rng = np.random.default_rng(8)
    w, dx = weights(rng, rehip.Q6_K, m, n), B.from_array(synth.activations(rng, rows, n))
    got = []
    for packed in (True, False):
        q = rehip.QMat.from_bytes(rehip.Q6_K, w, m, n)
        s, y = hip.Stream(), B(rows * m * 4)
        with pytest.MonkeyPatch.context() as mp:
            if not packed:
                mp.setenv("REHIP_GEMM_PACKED", "0")
            q.matmul_dev(dx, rows, y, rehip.MODE_BF16, stream=s)
            g = hip.Graph(s, lambda: q.matmul_dev(dx, rows, y, rehip.MODE_BF16, stream=s))
        g.launch()
        hip.synchronize()
        got.append(y.download(np.float32, rows * m))
        g.destroy()
        s.destroy()
        q.close()
    assert np.array_equal(got[0], got[1])
