"""Attention of 64 lanes and more needs no room that a call would have to find.

Its partials, where a launch cuts its tiles into segments, live in an array the
desk holds from its opening: a call neither grows the desk's workspace (which a
recording or a live replay refuses, and which moves the desk's generation) nor
writes the per-GPU array that calls of fewer lanes through
igl_attend_lanes_fixed_dev share.
"""
import ctypes

import numpy as np
import pytest

from igllm_amd import native
from igllm_amd.backend import Backend

pytestmark = pytest.mark.gpu

FIXED_FLOATS = 1 << 21
SCALE = 4.0 / 127.0


@pytest.fixture()
def desk():
    b = Backend(device=0, sum_limit=1024, col_limit=16384, lane_limit=16)
    yield b
    b.close()


def attend(b, entry, rings, ring, head, query, stride, lanes, place, out_ptr):
    return getattr(b.lib, entry)(ctypes.byref(b.desk), rings[0].ptr, rings[1].ptr, native.IGL_CACHE_INT8, SCALE, SCALE,
                                 ring, 1, 8, head, query, stride, place, 0, lanes, 1.0 / 16, out_ptr)


# five segments, more than one and one
@pytest.mark.parametrize("lanes,place,head", [(100, 1900, 256), (64, 8000, 512), (130, 0, 512), (1030, 0, 512)])
def test_wide_attention_needs_no_room(desk, lanes, place, head):
    print("case wide room", lanes, place, head, flush=True)
    lib, rng = desk.lib, np.random.default_rng(lanes)
    ring, stride = place + lanes, 8 * head
    rings = [desk.upload(rng.integers(0, 256, size=(ring, head), dtype=np.uint8)) for _ in range(2)]
    query = desk.upload(rng.normal(size=(lanes, stride)).astype(np.float32))
    out, lone = desk.alloc(lanes * stride * 4), desk.alloc(lanes * stride * 4)
    # each lane alone, first: its chunks' partials are all the workspace there is
    picks = sorted({0, 1, lanes // 2, lanes - 1})
    for lane in picks:
        at = 4 * stride * lane
        assert attend(desk, "igl_attend_lanes_dev", rings, ring, head, query.ptr + at, stride, 1, place + lane,
                      lone.ptr + at) == native.IGL_OKAY
    gate = desk.upload(np.ones(64, np.float32))
    desk.record_begin()
    assert lib.igl_gelu_gate_dev(ctypes.byref(desk.desk), gate.ptr, gate.ptr, 64) == native.IGL_OKAY
    replay = desk.record_end()
    before = lib.igl_desk_generation(ctypes.byref(desk.desk))
    shared = lib.igl_attend_fixed_ptr
    shared.restype, shared.argtypes = ctypes.c_void_p, [ctypes.c_int]
    fill = np.arange(FIXED_FLOATS, dtype=np.uint32)
    desk._check(lib.igl_copy_to_dev(ctypes.byref(desk.desk), shared(0), fill.ctypes.data, fill.nbytes), "copy_to_dev")
    got = []
    try:
        for entry in ("igl_attend_lanes_dev", "igl_attend_lanes_fixed_dev"):
            out.put(np.zeros(lanes * stride, np.float32))
            assert attend(desk, entry, rings, ring, head, query.ptr, stride, lanes, place, out.ptr) == native.IGL_OKAY
            desk.sync()
            got.append(out.get(np.float32, lanes * stride).reshape(lanes, stride))
    finally:
        desk.replay_free(replay)
    assert lib.igl_desk_generation(ctypes.byref(desk.desk)) == before
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    one = lone.get(np.float32, lanes * stride).reshape(lanes, stride)
    for lane in picks:
        err = float(np.max(np.abs(got[0][lane] - one[lane])))
        assert err <= 1e-5 * float(np.max(np.abs(one[lane]))) + 1e-7, (lane, err)
    kept = np.empty_like(fill)
    desk._check(lib.igl_copy_to_host(ctypes.byref(desk.desk), kept.ctypes.data, shared(0), kept.nbytes), "copy_to_host")
    assert np.array_equal(kept, fill)
    for b in rings + [query, out, lone, gate]:
        b.free()
