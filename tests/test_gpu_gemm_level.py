"""The integer GEMM of calibrated planes (five lanes and more) against each
lane's own launch.

One lane takes the level GEMV, whose sums are the reference's to the bit
(test_plane_lift_level_bitexact); every sum of the GEMM is an exact integer and
its row close the same, so the outputs are equal, bit for bit, whatever the
tile or the K slices.
"""
import ctypes

import numpy as np
import pytest

from igllm_amd.backend import Backend, make_plane

pytestmark = pytest.mark.gpu


# each tile's edges (64 x 64, 64 x 128, 128 x 128, 256 x 192: lanes x rows; in
# every width all four, with more steps than the stages: test_gemm_plan), K
# slices, one step, lanes below and past the GEMM's former floor
CASES = [(16, 128, 5), (300, 2048, 63), (96, 6144, 64), (1000, 256, 65), (4112, 384, 767), (6160, 128, 1030),
         (12304, 128, 1990), (4100, 640, 1000), (8100, 640, 2000), (12304, 640, 1990)]


@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("N,K,lanes", CASES)
def test_lanes_equal_single_lanes(backend, bits, N, K, lanes):
    rng = np.random.default_rng(N + K + lanes + bits)
    codes = rng.integers(0, 256, size=(N, (K * bits // 8 + 15) // 16 * 16), dtype=np.uint8)
    gains = (rng.random((N, 1)) * 0.02 + 0.01).astype(np.float32)
    cp = make_plane(codes, gains, K, group_size=K, bits=bits)
    cp.plane.enter_gain, cp.plane.leave_gain = 0.04, 0.1 * 4 ** (bits // 4)
    backend.attach(cp)
    act = rng.normal(size=(lanes, K + 4)).astype(np.float32)
    dev_act, out, one = backend.upload(act), backend.alloc(lanes * (N + 4) * 4), backend.alloc(N * 4)

    class Lane:
        ptr = 0

    backend.plane_lift_dev(cp, dev_act, K + 4, lanes, out, N + 4)
    backend.sync()
    got = out.get(np.float32, lanes * (N + 4)).reshape(lanes, N + 4)[:, :N]
    for lane in sorted({0, 1, 15, 16, 63, 64, lanes // 2, lanes - 1} & set(range(lanes))):
        Lane.ptr = dev_act.ptr + 4 * (K + 4) * lane
        backend.plane_lift_dev(cp, Lane, K, 1, one, N)
        backend.sync()
        assert np.array_equal(got[lane].view(np.uint32), one.get(np.float32, N).view(np.uint32)), lane
    for b in (dev_act, out, one):
        b.free()
    backend.detach(cp)


def test_few_lanes_grow_nothing():
    """The workspace of 5 to 63 lanes is reserved with the plane: a first lift,
    whatever its lanes, reallocates nothing (the desk's generation stays), and
    a live replay changes no bit of it."""
    b = Backend(device=0, sum_limit=1024, col_limit=16384, lane_limit=16)
    try:
        N, K = 96, 6144  # K in slices: the most workspace
        rng = np.random.default_rng(3)
        codes = rng.integers(0, 256, size=(N, K // 2), dtype=np.uint8)
        cp = make_plane(codes, np.full((N, 1), 0.02, np.float32), K, group_size=K)
        cp.plane.enter_gain, cp.plane.leave_gain = 0.04, 0.1
        b.attach(cp)
        act, out = b.upload(rng.normal(size=(63, K)).astype(np.float32)), b.alloc(63 * N * 4)
        before = b.lib.igl_desk_generation(ctypes.byref(b.desk))
        got = []
        for lanes in (5, 37, 63):
            b.plane_lift_dev(cp, act, K, lanes, out, N)
            b.sync()
            got.append(out.get(np.float32, lanes * N))
        b.record_begin()
        b.plane_lift_dev(cp, act, K, 37, out, N)
        replay = b.record_end()
        for lanes, want in zip((5, 37, 63), got):
            out.put(np.zeros(63 * N, np.float32))
            b.plane_lift_dev(cp, act, K, lanes, out, N)
            b.sync()
            assert np.array_equal(out.get(np.float32, lanes * N).view(np.uint32), want.view(np.uint32))
        b.replay_run(replay)
        b.sync()
        assert np.array_equal(out.get(np.float32, 37 * N).view(np.uint32), got[1].view(np.uint32))
        b.replay_free(replay)
        assert b.lib.igl_desk_generation(ctypes.byref(b.desk)) == before
        b.detach(cp)
        act.free()
        out.free()
    finally:
        b.close()
