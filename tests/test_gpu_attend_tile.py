"""Tiles of lanes (attend_tile_kernel) against each lane's own launch.

igl_attend_lanes_dev takes tiles of two or four lanes where their spans pass 64
positions; one lane alone always takes the chunk workgroups and their fold.
The two add the same terms in another order: bar 1e-5 max|o| + 1e-7, that of
the wide launches' test.
"""
import ctypes
import math

import numpy as np
import pytest

import oracle_lib as ol
from igllm_amd import native

pytestmark = pytest.mark.gpu


# ragged last tiles, chunks and segments; windows cut mid-tile; rings that wrap
# inside a chunk and rings no longer than the window; lanes that see nothing of
# a segment; tiles of four (more than 512 pairs); queries off 16-byte alignment
@pytest.mark.parametrize("lanes,window,place,head,fmt,kv,ring,pad", [
    (2, 0, 64, 512, 0, 1, 66, 0),
    (3, 0, 700, 512, 1, 1, 900, 0),
    (7, 70, 400, 512, 0, 1, 70, 0),
    (63, 65, 0, 512, 0, 1, 127, 0),
    (63, 0, 3000, 256, 1, 1, 3063, 1),
    (17, 512, 5000, 256, 0, 4, 530, 0),
    (65, 0, 0, 256, 0, 1, 65, 0),
    (129, 100, 777, 512, 0, 2, 228, 1),
    (90, 0, 2500, 256, 0, 1, 2590, 0),
    (515, 80, 60, 256, 1, 2, 595, 0),
    (1030, 0, 0, 512, 0, 1, 1030, 0),
])
def test_tiles_match_single_lanes(backend, lanes, window, place, head, fmt, kv, ring, pad):
    print("case tile", lanes, window, place, head, fmt, kv, ring, pad, flush=True)
    rng = np.random.default_rng(lanes + place)
    scale = 6.0 / 448.0 if fmt == 0 else 4.0 / 127.0
    rings = [backend.upload(ol.encode(np.clip(rng.normal(size=(ring, kv * head)), -4, 4).astype(np.float32), scale, fmt))
             for _ in range(2)]
    stride = 8 * kv * head + pad
    query = backend.upload(rng.normal(size=(lanes, stride)).astype(np.float32))
    out, one = backend.alloc(lanes * stride * 4), backend.alloc(8 * kv * head * 4)
    out.put(np.zeros(lanes * stride, np.float32))
    form = native.IGL_CACHE_INT8 if fmt else native.IGL_CACHE_E4M3

    def attend(query_ptr, at, count, out_ptr):
        rc = backend.lib.igl_attend_lanes_dev(
            ctypes.byref(backend.desk), rings[0].ptr, rings[1].ptr, form, scale, scale, ring, kv, 8, head, query_ptr,
            stride, at, window, count, 1.0 / math.sqrt(head), out_ptr)
        assert rc == native.IGL_OKAY, rc
        backend.sync()

    try:
        attend(query.ptr, place, lanes, out.ptr)
        got = out.get(np.float32, lanes * stride).reshape(lanes, stride)[:, :8 * kv * head]
        for lane in sorted({0, 1, 2, 3, 4, lanes // 2, lanes - 2, lanes - 1} & set(range(lanes))):
            attend(query.ptr + 4 * stride * lane, place + lane, 1, one.ptr)
            want = one.get(np.float32, 8 * kv * head)
            err = float(np.max(np.abs(got[lane] - want)))
            assert err <= 1e-5 * float(np.max(np.abs(want))) + 1e-7, (lane, err)
    finally:
        for b in rings + [query, out, one]:
            b.free()
