"""GPU parity: the reference scheme's tiled main pass (sage_ref_tile), at the
edges of its tiles: blocks below, at and past 16, 32, 64 and 128 keys (the
last on the per-row kernel), head dims around 64 and 128, a last block of one
key, fewer tokens than a block, queries that end inside a wave.  Every f32
operation keeps the reference's order and the INT8 products are exact, so the
device and the oracle's restatement agree bit for bit."""
import numpy as np
import pytest

from conftest import same

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    from quantibbler_amd import GpuContext

    return GpuContext(0)


def run(ctx, orc, q, k, v, causal, block):
    from quantibbler_amd import AttentionShape

    b, h, s, d = q.shape
    print("sage tile", q.shape, k.shape, v.shape, causal, block, flush=True)
    got = ctx.attention_sage(AttentionShape(b, h, k.shape[1], s, s, d, v.shape[3]), q, k, v, causal, block)
    want = orc.attention_sage_dev(q, k, v, causal, block).ravel()
    return np.asarray(got).ravel(), want


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,hk,s,d,dv,block", [
    (1, 2, 1, 1, 64, 64, 64), (1, 2, 2, 15, 64, 64, 16), (2, 4, 2, 65, 64, 64, 64), (1, 8, 8, 130, 128, 128, 64),
    (1, 2, 1, 193, 128, 128, 32), (1, 2, 2, 129, 128, 128, 128), (1, 2, 1, 300, 128, 64, 128),
    (1, 2, 1, 70, 20, 36, 24),    # 24 keys a block: a wave's queries end at different blocks
    (1, 3, 1, 77, 66, 130, 16),   # a value dim past the tile's: the per-row kernel
    (1, 2, 1, 90, 68, 100, 5), (1, 1, 1, 260, 100, 7, 100), (1, 2, 1, 40, 128, 128, 4096),
    (1, 1, 1, 140, 64, 64, 129),  # a block past 128 keys: the per-row kernel
])
def test_tiled_reference_scheme_bit_identical(ctx, orc, b, h, hk, s, d, dv, block, causal):
    rng = np.random.default_rng(1000 * s + block)
    q = rng.standard_normal((b, h, s, d)).astype(np.float32)
    k = (rng.standard_normal((b, hk, s, d)) + 2.0 * rng.standard_normal((b, hk, 1, d))).astype(np.float32)
    v = rng.standard_normal((b, hk, s, dv)).astype(np.float32)
    got, want = run(ctx, orc, q, k, v, causal, block)
    same(got, want)


@pytest.mark.parametrize("block", [16, 32, 64, 128])
def test_tiled_reference_scheme_extreme_values(ctx, orc, block):
    """Scores far apart (every p but one underflows), a zero query, zero keys
    and values, and an infinite key entry: its block's scores are NaN, which
    never win the maximum, and the rows that see them are NaN in both."""
    rng = np.random.default_rng(block)
    b, h, s, d = 1, 2, 150, 64
    q = (200.0 * rng.standard_normal((b, h, s, d))).astype(np.float32)
    k = (50.0 * rng.standard_normal((b, h, s, d))).astype(np.float32)
    v = rng.standard_normal((b, h, s, d)).astype(np.float32)
    q[0, 0, 3] = 0.0
    k[0, 0, :block] = 0.0
    v[0, 1, :block] = 0.0
    got, want = run(ctx, orc, q, k, v, True, block)
    same(got, want)
    k[0, 1, 140, 5] = np.inf
    got, want = run(ctx, orc, q, k, v, True, block)
    nan = np.isnan(want)
    assert nan.any() and not nan.all()
    assert np.array_equal(np.isnan(got), nan)
    same(got[~nan], want[~nan])
