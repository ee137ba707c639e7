"""A whole FFN over several rows (re_ffn_block_dev): the packed path (REHIP_GEMM_PACKED=2: at every shape
it takes) against an f64 FFN at the edges of its tiles and fragments, and against the separate calls.

Bounds: a bf16-mode product is off by 2^-7 + 2^-16 of sum |w x|, an f32-mode one by 3 * 2^-16 (split
operands), either by K * 2^-24 more for the f32 sums. |silu'| <= 1.1, so an error dg, du of the two
products moves h by 1.1 |dg| |u| + |silu(g)| |du| + 1.1 |dg| |du|, and SwiGLU in f32 by a few 2^-24."""
import numpy as np
import pytest

import oracle as O
import rehip
from rehip import hip, synth

pytestmark = pytest.mark.gpu
B = hip.DeviceBuffer
MODES = [rehip.MODE_BF16, rehip.MODE_F32]


def matrices(rng, t, td, d, ff):
    return [synth.weight_bytes(rng, t, ff, d), synth.weight_bytes(rng, t, ff, d), synth.weight_bytes(rng, td, d, ff)]


def block(q, x, rows, d, mode, add=None, in_place=False):
    f = rehip.Ffn(q[0], q[1])
    wb = f.block_work_bytes(q[2], rows)
    y = B.from_array(add) if in_place else B(rows * d * 4)
    a = None if add is None else y if in_place else B.from_array(add)
    f.block_dev(q[2], B.from_array(x), rows, y, B(wb), wb, mode, add=a)
    hip.synchronize()
    f.close()
    return y.download(np.float32, rows * d)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("t,td", [(rehip.Q4_0, rehip.Q8_0), (rehip.Q4_K, rehip.Q6_K), (rehip.Q5_0, rehip.Q5_K)])
@pytest.mark.parametrize("d,ff,rows", [(256, 256, 2), (512, 288, 65), (256, 544, 257), (896, 2080, 130), (512, 32, 33)])
def test_against_f64(t, td, d, ff, rows, mode, monkeypatch):
    monkeypatch.setenv("REHIP_GEMM_PACKED", "2")
    if td != rehip.Q8_0 and ff % 256:
        ff = -(-ff // 256) * 256                      # whole K-quant blocks
    if t != rehip.Q4_0 and t != rehip.Q5_0 and d % 256:
        d = -(-d // 256) * 256
    rng = np.random.default_rng(d + ff + rows)
    w = matrices(rng, t, td, d, ff)
    q = [rehip.QMat.from_bytes(t, w[0], ff, d), rehip.QMat.from_bytes(t, w[1], ff, d),
         rehip.QMat.from_bytes(td, w[2], d, ff)]
    x = (0.1 * synth.activations(rng, rows, d)).astype(np.float32)
    add = rng.standard_normal(rows * d).astype(np.float32)
    wg, wu = (O.dequant(t, b).reshape(ff, -1)[:, :d].astype(np.float64) for b in w[:2])
    wd = O.dequant(td, w[2]).reshape(d, -1)[:, :ff].astype(np.float64)
    xx = x.reshape(rows, d).astype(np.float64)
    eps = 2.0 ** -7 + 2.0 ** -16 if mode == rehip.MODE_BF16 else 3.01 * 2.0 ** -16
    g, u = xx @ wg.T, xx @ wu.T
    with np.errstate(over="ignore"):
        sg = g / (1 + np.exp(-g))
    dg, du = ((eps + d * 2.0 ** -24) * (np.abs(xx) @ np.abs(v).T) for v in (wg, wu))
    h = sg * u
    dh = 1.1 * dg * np.abs(u) + np.abs(sg) * du + 1.1 * dg * du + 2.0 ** -20 * np.abs(h)
    want = h @ wd.T
    bound = (dh + (eps + ff * 2.0 ** -24) * (np.abs(h) + dh)) @ np.abs(wd).T
    got = block(q, x, rows, d, mode)
    assert np.all(np.abs(got.reshape(rows, d) - want) <= bound)
    assert np.array_equal(block(q, x, rows, d, mode), got)
    plus = block(q, x, rows, d, mode, add)
    assert np.array_equal(plus, (add + got).astype(np.float32))
    assert np.array_equal(block(q, x, rows, d, mode, add, in_place=True), plus)
    for m in q:
        m.close()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("rows", [1, 5, 100, 300, 700])
def test_equals_separate_calls(mode, rows):
    """The default rule on both sides of its line: within the roundings of the separate calls, and their
    bits below 64 rows, where the block runs them."""
    d, ff = 224, 3072
    rng = np.random.default_rng(rows)
    w = matrices(rng, rehip.Q4_0, rehip.Q4_0, d, ff)
    q = [rehip.QMat.from_bytes(rehip.Q4_0, b, *s) for b, s in zip(w, ((ff, d), (ff, d), (d, ff)))]
    x = (0.1 * synth.activations(rng, rows, d)).astype(np.float32)
    add = rng.standard_normal(rows * d).astype(np.float32)
    dx, g, u, h, o = B.from_array(x), B(rows * ff * 4), B(rows * ff * 4), B(rows * ff * 4), B(rows * d * 4)
    q[0].matmul_dev(dx, rows, g, mode)
    q[1].matmul_dev(dx, rows, u, mode)
    rehip.swiglu_dev(g, u, h, rows * ff)
    q[2].matmul_dev(h, rows, o, mode)
    rehip.add_dev(B.from_array(add), o, rows * d, rows * d, o)
    hip.synchronize()
    want, got = o.download(np.float32, rows * d), block(q, x, rows, d, mode, add)
    assert np.linalg.norm(got - want) <= (1e-2 if mode == rehip.MODE_BF16 else 2e-5) * np.linalg.norm(want - add)
    if rows < 64:
        assert np.array_equal(got, want)
    for m in q:
        m.close()


@pytest.mark.parametrize("mode", MODES)
def test_one_matrix_as_gate_and_up(mode):
    """The packed path against the separate calls where gate and up are one matrix, after a call on other
    weights that leaves its packed groups in the shared workspace."""
    d, ff, rows = 256, 512, 150
    rng = np.random.default_rng(11)
    w = matrices(rng, rehip.Q4_K, rehip.Q6_K, d, ff)
    q = [rehip.QMat.from_bytes(t, b, *s) for t, b, s in zip((rehip.Q4_K, rehip.Q4_K, rehip.Q6_K), w,
                                                            ((ff, d), (ff, d), (d, ff)))]
    x = (0.1 * synth.activations(rng, rows, d)).astype(np.float32)
    got = []
    for knob in ("2", "0"):
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv("REHIP_GEMM_PACKED", knob)
            block(q, x, rows, d, mode)
            got.append(block([q[1], q[1], q[2]], x, rows, d, mode))
    # products in another order of sums: an h may round to bf16 the other way (2^-8 of it)
    assert np.linalg.norm(got[0] - got[1]) <= (2.0 ** -8 if mode == rehip.MODE_BF16 else 2e-5) * np.linalg.norm(got[1])
    for m in q:
        m.close()


def test_capture_after_eager_call_keeps_its_slices():
    """A captured FFN (separate calls) after an eager one on packed operands, at the row count that the
    few-row GEMM serves: its K slices, so the bits of separate calls that never packed."""
    d, ff, rows = 896, 4864, 64
    rng = np.random.default_rng(12)
    w = matrices(rng, rehip.Q4_K, rehip.Q6_K, d, ff)
    x = B.from_array((0.1 * synth.activations(rng, rows, d)).astype(np.float32))
    got = []
    for packed in (True, False):
        q = [rehip.QMat.from_bytes(t, b, *s) for t, b, s in zip((rehip.Q4_K, rehip.Q4_K, rehip.Q6_K), w,
                                                                ((ff, d), (ff, d), (d, ff)))]
        f = rehip.Ffn(q[0], q[1])
        wb = f.block_work_bytes(q[2], rows)
        y, wk, s = B(rows * d * 4), B(wb), hip.Stream()

        def call():
            f.block_dev(q[2], x, rows, y, wk, wb, rehip.MODE_F32, stream=s)
        with pytest.MonkeyPatch.context() as mp:
            if not packed:
                mp.setenv("REHIP_GEMM_PACKED", "0")
            call()
            g = hip.Graph(s, call)
        for _ in range(3):
            g.launch()
            hip.synchronize()
        got.append(y.download(np.float32, rows * d))
        g.destroy()
        s.destroy()
        f.close()
        for m in q:
            m.close()
    assert np.array_equal(got[0], got[1])


def test_errors():
    rng = np.random.default_rng(1)
    w = matrices(rng, rehip.Q4_0, rehip.Q4_0, 64, 96)
    q = [rehip.QMat.from_bytes(rehip.Q4_0, b, *s) for b, s in zip(w, ((96, 64), (96, 64), (64, 96)))]
    f = rehip.Ffn(q[0], q[1])
    x, y, wk = B(64 * 4 * 2), B(64 * 4 * 2), B(1 << 16)
    with pytest.raises(rehip.RehipError):
        f.block_dev(q[0], x, 2, y, wk, 1 << 16)                    # 64 columns for 96
    with pytest.raises(rehip.RehipError):
        f.block_dev(q[2], x, 2, y, wk, f.block_work_bytes(q[2], 2) - 4)
    with pytest.raises(rehip.RehipError):
        f.block_dev(q[2], x, 2, y, wk, 1 << 16, 7)
    f.close()
    for m in q:
        m.close()


@pytest.mark.parametrize("mode,d,ff,rows", [(rehip.MODE_F32, 1024, 11008, 9728), (rehip.MODE_BF16, 1024, 24576, 8960),
                                            (rehip.MODE_F32, 8192, 4096, 8704)])
def test_weights_in_pieces(mode, d, ff, rows):
    """x and h fill most of the workspace: gate and up (and in the last case down) are packed and
    multiplied in pieces. Some rows of the result against the same rows in a call of their own."""
    rng = np.random.default_rng(9)
    w = matrices(rng, rehip.Q4_0, rehip.Q8_0, d, ff)
    q = [rehip.QMat.from_bytes(t, b, *s) for t, b, s in zip((rehip.Q4_0, rehip.Q4_0, rehip.Q8_0), w,
                                                            ((ff, d), (ff, d), (d, ff)))]
    x = (0.1 * synth.activations(rng, rows, d)).astype(np.float32).reshape(rows, d)
    got = block(q, x, rows, d, mode).reshape(rows, d)
    for r0 in (0, rows - 300):
        part = block(q, x[r0:r0 + 300].copy(), 300, d, mode).reshape(300, d)
        diff = np.linalg.norm(got[r0:r0 + 300] - part, axis=1) / np.linalg.norm(part, axis=1)
        assert diff.max() <= (2e-3 if mode == rehip.MODE_BF16 else 1e-5)   # sums in another K split
    for m in q:
        m.close()
