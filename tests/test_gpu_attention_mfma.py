"""Prefill attention on f32 MFMAs (rows >= 8, head_dim 32 / 64 / 96 / 128) at its edges: part-filled
vector blocks (32 query vectors of a kv head) and key blocks (32 keys, eight waves), positions at the
cache's end, and non-finite values in rows that a query may not see."""
import numpy as np
import pytest

import rehip
from rehip import hip

pytestmark = pytest.mark.gpu
B = hip.DeviceBuffer


def reference(q, kc, vc, pos, kv_heads):
    """f64 causal GQA attention over exactly the rows each query sees."""
    rows, heads, hd = q.shape
    out = np.empty(q.shape)
    with np.errstate(invalid="ignore", over="ignore"):
        for r in range(rows):
            n = min(pos + r + 1, kc.shape[0])
            for h in range(heads):
                kv = h * kv_heads // heads
                s = kc[:n, kv].astype(np.float64) @ q[r, h].astype(np.float64) / np.sqrt(hd)
                p = np.exp(s - s.max())
                out[r, h] = (p / p.sum()) @ vc[:n, kv].astype(np.float64)
    return out


def run(q, kc, vc, pos):
    rows, heads, hd = q.shape
    ctx = B(q.nbytes)
    rehip.attention_dev(B.from_array(q), B.from_array(kc), B.from_array(vc), rows, heads, kc.shape[1], hd,
                        kc.shape[0], B.from_array(np.array([pos], np.int32)), ctx)
    hip.synchronize()
    return ctx.download(np.float32, q.size).reshape(q.shape)


@pytest.mark.parametrize("hd", [32, 64, 96, 128])
@pytest.mark.parametrize("rows,pos,heads,kv_heads,max_seq", [(8, 0, 1, 1, 8), (9, 23, 7, 1, 32), (33, 250, 6, 2, 300),
                                                             (31, 226, 3, 3, 257), (40, 480, 8, 1, 512)])
def test_edges(hd, rows, pos, heads, kv_heads, max_seq):
    """(40 rows at 480 of a 512-row cache: the last ones run past it and see its every row.)"""
    rng = np.random.default_rng(hd + rows)
    q = 2 * rng.standard_normal((rows, heads, hd)).astype(np.float32)
    kc, vc = (rng.standard_normal((max_seq, kv_heads, hd)).astype(np.float32) for _ in range(2))
    want = reference(q, kc, vc, pos, kv_heads)
    # scores of size <= 8 off by <= 64 roundings each, so probabilities by <= 64 * 8 * 2^-24 = 3e-5
    np.testing.assert_allclose(run(q, kc, vc, pos), want, rtol=0, atol=3e-5 * np.abs(want).max())


@pytest.mark.parametrize("hd,pairs", [(32, 400), (96, 600), (128, 900)])
def test_few_pairs_with_a_workspace_split_the_cache(hd, pairs):
    """On both sides of the line, with and without a workspace: the same attention, and the workspace used
    (its splits written) up to the line only."""
    heads, kv_heads, max_seq, pos = 10, 2, 300, 200
    rng = np.random.default_rng(hd)
    kc, vc = (rng.standard_normal((max_seq, kv_heads, hd)).astype(np.float32) for _ in range(2))
    for rows in (8, pairs // heads, pairs // heads + 1):
        q = 2 * rng.standard_normal((rows, heads, hd)).astype(np.float32)
        wb = rehip.attention_work_bytes(rows, heads, hd, max_seq)
        work, ctx = B.from_array(np.full(wb // 4, 7.5, np.float32)), B(q.nbytes)
        rehip.attention_dev(B.from_array(q), B.from_array(kc), B.from_array(vc), rows, heads, kv_heads, hd, max_seq,
                            B.from_array(np.array([pos], np.int32)), ctx, work=work, work_bytes=wb)
        hip.synchronize()
        assert np.any(work.download(np.float32, wb // 4) != 7.5) == (rows * heads <= pairs)
        want = reference(q, kc, vc, pos, kv_heads)
        tol = 3e-5 * np.abs(want).max()
        np.testing.assert_allclose(ctx.download(np.float32, q.size).reshape(q.shape), want, rtol=0, atol=tol)
        np.testing.assert_allclose(run(q, kc, vc, pos), want, rtol=0, atol=tol)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_hidden_rows_may_hold_anything(hd, bad):
    """A row's K and V reach the queries from that row on and no earlier one, whatever they hold."""
    rng = np.random.default_rng(hd)
    q = rng.standard_normal((50, 4, hd)).astype(np.float32)
    kc, vc = (rng.standard_normal((128, 2, hd)).astype(np.float32) for _ in range(2))
    vc[40 + 27, 1, 5] = bad
    kc[40 + 45, 0] = bad
    vc[90:], kc[90:] = bad, bad
    want, got = reference(q, kc, vc, 40, 2), run(q, kc, vc, 40)
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(want))
    fine = np.isfinite(want)
    np.testing.assert_allclose(got[fine], want[fine], rtol=0, atol=3e-5 * np.abs(want[fine]).max())
