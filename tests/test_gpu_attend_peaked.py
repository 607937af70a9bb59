"""Attention whose scores are not flat: a sink position far above the others,
and a lane whose query holds a NaN.

A trained model puts most of a head's weight on one early position.  The
others' weights are then e^-10 to e^-18 of it, and where the sink's own value
is small they make the blend: their relative error has to stay that of flat
scores.  Bars are sums of the kernels' roundings (u = 2^-24):
- a score: 24 additions at most of sum |q k|, the query's two terms 2;
- a weight: its score and the sink's, three exponentials (argument, log2 e,
  result) of arguments up to the scores' range;
- a weight's two binary16 terms: 2 u of it, and half a subnormal step (u) of
  the largest weight in its chunk (the sink's chunk holds no other value, so
  the sink's size is no allowance for the other chunks);
- the blend: 24 additions in a chunk, 3 a chunk after it.
"""
import ctypes
import math

import numpy as np
import pytest

import oracle_lib as ol
from igllm_amd import native

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def decode(rows, scale, fmt):
    grid = ol.grid_i8(scale) if fmt else ol.grid8(scale)
    return np.asarray(grid, np.float64)[rows]


def attend(backend, rings, fmt, scale, ring, head, query, lanes, place, window, out):
    rc = backend.lib.igl_attend_lanes_dev(
        ctypes.byref(backend.desk), rings[0].ptr, rings[1].ptr, native.IGL_CACHE_INT8 if fmt else native.IGL_CACHE_E4M3,
        scale, scale, ring, 1, 8, head, query.ptr, 8 * head, place, window, lanes, 1.0 / math.sqrt(head), out.ptr)
    assert rc == native.IGL_OKAY, rc
    backend.sync()
    return out.get(np.float32, lanes * 8 * head).reshape(lanes, 8, head)


# tiles of two and four lanes, cut into segments and not; the chunk workgroups
# (one lane); the value of the sink and its chunk zero, and one like the others'
@pytest.mark.parametrize("value", [0.0, 1.0])
@pytest.mark.parametrize("peak", [10.0, 18.0])
@pytest.mark.parametrize("lanes,place,head,fmt", [
    (1, 1999, 256, 1), (2, 300, 512, 0), (32, 4000, 512, 1), (100, 1900, 256, 0), (130, 0, 512, 1), (600, 0, 512, 0),
    (1030, 0, 512, 0), (1100, 900, 256, 1),
])
def test_sink(backend, lanes, place, head, fmt, peak, value):
    print("case sink", lanes, place, head, fmt, peak, value, flush=True)
    rng = np.random.default_rng(lanes + place)
    ring, flat = place + lanes, 32  # dims only the sink's key has
    scale = 4.0 / 127.0 if fmt else 6.0 / 448.0
    key, val = (np.clip(rng.normal(size=(ring, head)), -4, 4).astype(np.float32) for _ in range(2))
    key[:, :flat] = 0.0
    key[0] = 0.0
    key[0, :flat] = 4.0
    val[:64] = value * val[:1]
    key, val = ol.encode(key, scale, fmt), ol.encode(val, scale, fmt)
    query = rng.normal(size=(lanes, 8, head)).astype(np.float32)
    query[:, :, :flat] = peak * math.sqrt(head) / (4.0 * flat)
    rings = [backend.upload(key), backend.upload(val)]
    q_dev, out = backend.upload(query), backend.alloc(query.nbytes)
    try:
        got = attend(backend, rings, fmt, scale, ring, head, q_dev, lanes, place, 0, out)
    finally:
        for b in rings + [q_dev, out]:
            b.free()
    key, val = decode(key, scale, fmt), decode(val, scale, fmt)
    for lane in sorted({0, 1, lanes // 2, lanes - 1} & set(range(lanes))):
        n = place + lane + 1
        k, v, q = key[:n], val[:n], query[lane].astype(np.float64)
        score = q @ k.T / math.sqrt(head)
        size = np.abs(q) @ np.abs(k).T / math.sqrt(head)
        w = np.exp(score - score.max(1, keepdims=True))
        reach = score.max(1, keepdims=True) - score.min(1, keepdims=True)
        top = np.stack([w[:, c:c + 64].max(1) for c in range(0, n, 64)], 1).repeat(64, 1)[:, :n]
        each = w * (26 * (size + size[:, :1]) + 6 * reach + 8 + 24 + 3 * (n / 64 + 1)) + 2 * w + top
        total = w.sum(1, keepdims=True)
        err = np.abs(got[lane] - w @ v / total)
        bound = U * (each @ np.abs(v)) / total
        assert np.all(err <= bound), (lane, float((err / bound).max()))


# tiles, and tiles folded from segments
@pytest.mark.parametrize("lanes,place,head", [(16, 300, 512), (100, 1900, 256), (130, 0, 512), (600, 0, 512),
                                              (1030, 0, 512)])
def test_nan_query(backend, lanes, place, head):
    """A NaN in one head of one lane's query: that head's blend is NaN,
    whatever form the launch takes, and no other output changes."""
    print("case nan query", lanes, place, head, flush=True)
    rng = np.random.default_rng(lanes)
    ring, scale = place + lanes, 4.0 / 127.0
    rings = [backend.upload(rng.integers(0, 256, size=(ring, head), dtype=np.uint8)) for _ in range(2)]
    query = rng.normal(size=(lanes, 8, head)).astype(np.float32)
    lane = lanes // 2
    bad = query.copy()
    bad[lane, 3, 7] = np.nan
    q_dev, bad_dev, out = backend.upload(query), backend.upload(bad), backend.alloc(query.nbytes)
    try:
        want = attend(backend, rings, 1, scale, ring, head, q_dev, lanes, place, 0, out)
        got = attend(backend, rings, 1, scale, ring, head, bad_dev, lanes, place, 0, out)
    finally:
        for b in rings + [q_dev, bad_dev, out]:
            b.free()
    assert np.isnan(got[lane, 3]).all(), got[lane, 3, :4]
    got[lane, 3] = want[lane, 3]
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
