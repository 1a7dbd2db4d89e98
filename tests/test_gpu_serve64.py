"""GPU parity: fp32 serving's f64 products (serve64.hip) bit for bit against the
oracle's element-order sums, at the edges of the kernel's tiles: 16-row groups,
128-wide slices, chunks of 16 slices (2048 k), and single rows and columns."""
import numpy as np
import pytest

from conftest import same

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    from quantibbler_amd import GpuContext

    return GpuContext(0)


def layer(ctx, orc, rng, dout, din, r):
    from quantibbler_amd import FactorLayer

    ub = orc.pack_bits(rng.choice([-1, 1], (dout, r)).astype(np.int8))
    vt = orc.pack_bits(rng.choice([-1, 1], (r, din)).astype(np.int8))
    s1 = np.exp(0.5 * rng.standard_normal(dout)).astype(np.float32)
    s2 = np.exp(0.5 * rng.standard_normal(din)).astype(np.float32)
    bias = rng.standard_normal(dout).astype(np.float32)
    return FactorLayer.from_rows(ctx, dout, din, r, ub, vt, s1, s2, bias), (ub, vt, s1, s2, bias)


@pytest.mark.parametrize("dout,din,r", [
    (1, 1, 1), (15, 127, 17), (16, 128, 16), (17, 129, 127), (130, 2047, 128), (48, 2048, 129), (33, 2049, 40),
    (20, 4200, 2100), (300, 640, 1),
])
def test_fp32_products_bit_identical(ctx, orc, dout, din, r):
    print("serve64", dout, din, r, flush=True)
    rng = np.random.default_rng(dout + 7 * din + r)
    L, p = layer(ctx, orc, rng, dout, din, r)
    x = rng.standard_normal((2, din)).astype(np.float32)
    # the second token's entries span 2^80: sums whose every rounding depends on the order
    x[1] *= (2.0 ** rng.uniform(-40, 40, din)).astype(np.float32)
    got = L.apply(x, "float32")
    for i in range(2):
        same(got[i], orc.factor_apply("fp32", dout, din, r, *p, x[i]))


def test_fp32_products_with_infinities(ctx, orc):
    """An infinite activation gives the oracle's infinities and NaNs."""
    rng = np.random.default_rng(9)
    L, p = layer(ctx, orc, rng, 40, 300, 50)
    x = rng.standard_normal(300).astype(np.float32)
    x[100] = np.inf
    got, want = L.apply(x, "float32"), orc.factor_apply("fp32", 40, 300, 50, *p, x)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    same(got[~np.isnan(want)], want[~np.isnan(want)])
