"""The matrix-core product of real planes (bf16 and binary16 rows, five lanes
and more) against the 64-bit product of the same values.

Every term product is exact, so an output's error is the rounding of its fp32
additions: a product passes at most 16 inside its chain of four 32-wide steps,
K / 128 as the finished chains are added, and 15 more across the waves' K
split, each at most half an ulp of a sum no larger than sum |x w|.
"""
import numpy as np
import pytest

from igllm_amd import native
from igllm_amd.backend import CodePlane
from igllm_amd.native import Plane

pytestmark = pytest.mark.gpu


def bf16_bits(x):
    return (x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)  # truncated: any bf16 values do


def product(backend, kind, N, K, lanes, act, rows, stride):
    p = Plane()
    p.row_count, p.col_count, p.form = N, K, native.IGL_PLANE_REAL
    p.real_type = native.IGL_STORE_BF16 if kind == "bf16" else native.IGL_STORE_F16
    p.real_data = rows.ctypes.data
    cp = backend.attach(CodePlane(p, rows, None))
    dev_act, dev_out = backend.upload(act), backend.alloc(lanes * (N + 3) * 4)
    backend.mat_mat_dev(cp, dev_act, stride, lanes, dev_out, N + 3)
    backend.sync()
    out = dev_out.get(np.float32, lanes * (N + 3)).reshape(lanes, N + 3)[:, :N]
    dev_act.free()
    dev_out.free()
    backend.detach(cp)
    return out


def case(kind, N, K, lanes, seed, spread=False):
    rng = np.random.default_rng(seed)
    w = (rng.normal(size=(N, K)) * 0.02).astype(np.float32)
    stride = K + 4
    act = rng.normal(size=(lanes, stride)).astype(np.float32)
    if spread:  # the terms' whole exponent range
        act *= np.exp2(rng.integers(-60, 60, size=act.shape)).astype(np.float32)
    rows = bf16_bits(w) if kind == "bf16" else w.astype(np.float16)
    value = (rows.astype(np.uint32) << 16).view(np.float32) if kind == "bf16" else rows
    return act, rows, value.astype(np.float64), stride


# every tile form's edges: 16 x 16, 32 x 16 (one and two a CU), 32 x 32, 64 x
# 32, 64 x 64 split and unsplit (test_gemm_plan checks that all are seen); K of
# one step, and not a whole K split
CASES = [(1, 32, 5), (17, 96, 17), (300, 288, 15), (4100, 352, 16), (8193, 64, 13), (4097, 160, 33), (8190, 96, 31),
         (4090, 544, 65), (8960, 1536, 70), (16, 2048, 500), (4100, 1056, 16), (8193, 1568, 13), (8190, 1056, 31),
         (8960, 1536, 64), (8950, 544, 48)]


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("N,K,lanes", CASES)
@pytest.mark.parametrize("spread", [False, True])
def test_real_product(backend, kind, N, K, lanes, spread):
    act, rows, value, stride = case(kind, N, K, lanes, N + K + lanes, spread)
    got = product(backend, kind, N, K, lanes, act, rows, stride)
    x = act[:, :K].astype(np.float64)
    bound = (16 + K / 128 + 15 + 2) * 2.0 ** -24 * (np.abs(x) @ np.abs(value).T)
    assert np.all(np.abs(got - x @ value.T) <= bound)


# 16 x 16 and 64 x 64, K split eight and four ways, and 64 x 64 unsplit
@pytest.mark.parametrize("N,lanes", [(70, 20), (8960, 48), (4100, 500)])
@pytest.mark.parametrize("kind", ["bf16", "f16"])
def test_real_product_of_infinities(backend, kind, N, lanes):
    """An infinite or NaN operand gives what the FMAs of a row give, and
    leaves the other outputs alone; the largest finite activations have three
    finite terms."""
    K = 256
    act, rows, value, stride = case(kind, N, K, lanes, 3)
    want = act[:, :K].astype(np.float64) @ value.T
    act[2, 5], act[7, 100], act[11, 255] = np.inf, -np.inf, np.nan
    act[13, :K] = 0.0
    act[13, 17] = np.float32(3.4e38)
    rows[9, 40] = 0x7F80 if kind == "bf16" else np.float16(np.inf)
    value = ((rows.astype(np.uint32) << 16).view(np.float32) if kind == "bf16" else rows).astype(np.float64)
    got = product(backend, kind, N, K, lanes, act, rows, stride)
    x = act[:, :K].astype(np.float64)
    for m in (2, 7, 11):
        for n in (0, 9, 69):
            full = x[m] * value[n]
            total = np.nan if np.isnan(full).any() else full.sum()
            assert np.array_equal(got[m, n], np.float32(total), equal_nan=True), (m, n)
    big = np.float64(act[13, 17]) * value[:, 17]
    big[9] = np.nan  # 0 x inf
    assert np.allclose(got[13], big, rtol=2.0 ** -22, atol=0, equal_nan=True)
    rest = [m for m in range(lanes) if m not in (2, 7, 11, 13)]
    keep = [n for n in range(N) if n != 9]
    assert np.array_equal(got[rest, 9], np.float32(np.sign(x[rest, 40]) * np.inf))
    assert np.allclose(got[np.ix_(rest, keep)], want[np.ix_(rest, keep)], rtol=0, atol=1e-5)


# K split eight and four ways, and not
@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("N,K,lanes", [(300, 512, 12), (8960, 544, 48), (2560, 96, 512)])
def test_real_product_of_small_activations(backend, kind, N, K, lanes):
    """Lanes of activations near the three terms' last bit (2^-133) and below,
    where an output is formed again by FMAs: K additions at most, and half of
    2^-149 each where they are subnormal."""
    act, rows, value, stride = case(kind, N, K, lanes, 5)
    for lane, scale in ((1, 2.0 ** -112), (2, 2.0 ** -119), (3, 2.0 ** -128), (4, 0.0)):
        act[lane] *= np.float32(scale)
    got = product(backend, kind, N, K, lanes, act, rows, stride)
    x = act[:, :K].astype(np.float64)
    bound = (K + 2) * (2.0 ** -24 * (np.abs(x) @ np.abs(value).T) + 2.0 ** -150)
    bound[5:] = (16 + K / 128 + 15 + 2) * 2.0 ** -24 * (np.abs(x[5:]) @ np.abs(value).T)
    assert np.all(np.abs(got - x @ value.T) <= bound)
