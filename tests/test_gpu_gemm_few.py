"""The few-lane product of 4-bit planes (9 to 63 lanes) against the 64-bit
product of the same values.

Every product of a term and a code is exact, so an output's error is the
rounding of its fp32 additions: a product passes at most 12 inside its unit's
chain, the gain's multiply-add, seven more in a run of eight units, K / 1024
runs a wave (four waves share K at least), and 15 across the waves; each at
most half an ulp of a sum no larger than sum |x w|.  test_gemm_plan checks that
the cases take every tile.
"""
import numpy as np
import pytest

from igllm_amd.backend import make_plane

pytestmark = pytest.mark.gpu


# the tiles' edges, K of one unit, not a whole K split, more than one run and
# more stages than the ring holds in every tile; wider groups and one gain a
# row; lanes and outputs with a stride
CASES = [
    (1, 32, 9, 32), (17, 96, 63, 32), (4097, 64, 15, 32), (8193, 128, 16, 64), (1000, 1056, 33, 32),
    (4100, 544, 31, 544), (6145, 1536, 49, 32), (8192, 2080, 63, 32), (12300, 96, 47, 96), (16400, 64, 63, 32),
    (300, 6176, 17, 128), (5000, 12288, 12, 32), (8193, 4128, 11, 32), (10000, 2336, 16, 32), (8190, 2336, 24, 32),
    (6144, 1536, 37, 32), (6150, 2336, 47, 32), (6140, 2336, 63, 32), (12300, 1568, 63, 32),
]


@pytest.mark.parametrize("N,K,lanes,group", CASES)
@pytest.mark.parametrize("spread", [False, True])
def test_few_lanes(backend, N, K, lanes, group, spread):
    rng = np.random.default_rng(N + K + lanes)
    stride = (K // 2 + 15) // 16 * 16
    codes = rng.integers(0, 256, size=(N, stride), dtype=np.uint8)
    groups = (K + group - 1) // group
    gains = np.abs(rng.normal(0, 0.02, size=(N, groups))).astype(np.float32)
    act = rng.normal(size=(lanes, K + 4)).astype(np.float32)
    if spread:  # the terms' exponent range
        act *= np.exp2(rng.integers(-60, 60, size=act.shape)).astype(np.float32)
    cp = backend.attach(make_plane(codes, gains, K, group_size=group))
    dev_act, dev_out = backend.upload(act), backend.alloc(lanes * (N + 3) * 4)
    backend.gemv_dev(cp, dev_act, K + 4, lanes, dev_out, N + 3)
    backend.sync()
    got = dev_out.get(np.float32, lanes * (N + 3)).reshape(lanes, N + 3)[:, :N]
    dev_act.free()
    dev_out.free()
    backend.detach(cp)
    value = np.empty((N, K), np.float64)
    value[:, 0::2] = (codes[:, :K // 2] & 15).astype(np.float64) - 8
    value[:, 1::2] = (codes[:, :K // 2] >> 4).astype(np.float64) - 8
    value *= np.repeat(gains.astype(np.float64), group, axis=1)[:, :K]
    x = act[:, :K].astype(np.float64)
    bound = (12 + 2 + 7 + K / 1024 + 15) * 2.0 ** -24 * (np.abs(x) @ np.abs(value).T)
    assert np.all(np.abs(got - x @ value.T) <= bound)


# K split sixteen and eight ways, more than one wave row
@pytest.mark.parametrize("N,K,lanes", [(300, 512, 12), (4100, 544, 40), (12300, 96, 60)])
def test_few_lanes_activation_range(backend, N, K, lanes):
    """Lanes of activations near fp32's ends: unit sums past its range that
    their gains bring back, values below the three terms' last bit, subnormal
    ones, zero, infinite and NaN.  Formed again, an output passes its unit's 32
    additions and one a unit, a weight's rounding, and where it is subnormal
    half of 2^-149 a unit."""
    rng = np.random.default_rng(N)
    codes = rng.integers(0, 256, size=(N, K // 2), dtype=np.uint8)
    gains = np.abs(rng.normal(0, 0.02, size=(N, K // 32))).astype(np.float32)
    act = rng.normal(size=(lanes, K)).astype(np.float32)
    for lane, scale in ((1, 2.0 ** 123), (2, 2.0 ** -112), (3, 2.0 ** -119), (4, 2.0 ** -128), (5, 0.0)):
        act[lane] *= np.float32(scale)
    act[6, 3], act[7, K - 1], act[8, 40] = np.inf, -np.inf, np.nan
    cp = backend.attach(make_plane(codes, gains, K))
    dev_act, dev_out = backend.upload(act), backend.alloc(lanes * N * 4)
    backend.gemv_dev(cp, dev_act, K, lanes, dev_out, N)
    backend.sync()
    got = dev_out.get(np.float32, lanes * N).reshape(lanes, N)
    dev_act.free()
    dev_out.free()
    backend.detach(cp)
    value = np.empty((N, K), np.float64)
    value[:, 0::2] = (codes & 15).astype(np.float64) - 8
    value[:, 1::2] = (codes >> 4).astype(np.float64) - 8
    value *= np.repeat(gains.astype(np.float64), 32, axis=1)
    x = act.astype(np.float64)
    finite = [m for m in range(lanes) if m not in (6, 7, 8)]
    want = x[finite] @ value.T
    assert np.abs(want).max() < 3.4e38
    bound = (32 + 1 + K / 32 + 2) * 2.0 ** -24 * (np.abs(x[finite]) @ np.abs(value).T) + K / 32 * 2.0 ** -150
    assert np.all(np.abs(got[finite] - want) <= bound)
    for m, k in ((6, 3), (7, K - 1)):
        side = np.sign(value[:, k]) * np.sign(act[m, k])
        assert np.array_equal(got[m], np.where(side == 0, np.nan, side * np.inf).astype(np.float32), equal_nan=True)
    assert np.isnan(got[8]).all()
