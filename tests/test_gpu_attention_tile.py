"""GPU: the exact attention face on the f32 matrix cores (att_tile), at the
edges of its tiles (16 queries, 32 keys, 64-channel halves), against float64.

Tolerance: a score is a sum of d products, the output a weighted mean of at
most max|v|.  With eps = 2^-24 a score's error is at most (d / 2 + 4) eps
sum|q k| / sqrt(d) in the worst case and sqrt of that count in practice; the
bound below takes the worst case for the score (a relative error of p) and 64
eps max|v| for the weighted mean's blocked sums and exp."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")
EPS = 2.0 ** -24


@pytest.fixture(scope="module")
def ctx():
    from quantibbler_amd import GpuContext

    return GpuContext(0)


def reference(q, k, v, causal):
    """float64, masked keys left out altogether (their values may be anything)."""
    b, h, sq, d = q.shape
    hk, skv = k.shape[1], k.shape[2]
    out = np.full((b, h, sq, v.shape[3]), np.nan)
    bound = np.zeros(out.shape)
    for bi in range(b):
        for hi in range(h):
            K, V = k[bi, hi // (h // hk)].astype(np.float64), v[bi, hi // (h // hk)].astype(np.float64)
            for i in range(sq):
                n = min(skv, max(0, i + skv - sq + 1)) if causal else skv
                if n == 0:
                    continue
                x = q[bi, hi, i].astype(np.float64)
                s = K[:n] @ x / np.sqrt(d)
                with np.errstate(invalid="ignore"):
                    p = np.exp(s - s.max())
                    out[bi, hi, i] = (p @ V[:n]) / p.sum()
                score = (d / 2 + 4) * EPS * (np.abs(K[:n]) @ np.abs(x)).max() / np.sqrt(d)
                bound[bi, hi, i] = (2 * score + 64 * EPS) * np.abs(V[:n]).max()
    return out, bound


def run(ctx, q, k, v, causal):
    from quantibbler_amd import AttentionShape

    b, h, sq, d = q.shape
    print("attention tile", q.shape, k.shape, v.shape, causal, flush=True)
    sh = AttentionShape(b, h, k.shape[1], sq, k.shape[2], d, v.shape[3])
    return np.asarray(ctx.attention(sh, q, k, v, causal)).reshape(b, h, sq, v.shape[3])


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,hk,sq,skv,d,dv", [
    (1, 2, 1, 1, 1, 64, 64), (1, 2, 1, 1, 33, 128, 128), (2, 4, 2, 16, 32, 64, 64), (1, 4, 1, 17, 300, 128, 128),
    (1, 2, 2, 65, 65, 80, 48), (1, 2, 1, 33, 31, 16, 128),     # more queries than keys: rows with no key
    (1, 2, 1, 40, 700, 112, 80), (1, 40, 8, 130, 150, 64, 64),  # two query tiles a workgroup
    (2, 100, 50, 70, 40, 128, 128),                             # four
    (1, 2, 1, 20, 50, 20, 24),                                  # rows that are not whole steps: a row a workgroup
])
def test_tile_matches_float64(ctx, b, h, hk, sq, skv, d, dv, causal):
    rng = np.random.default_rng(100 * sq + skv + d)
    q = rng.standard_normal((b, h, sq, d)).astype(np.float32)
    k = (rng.standard_normal((b, hk, skv, d)) + rng.standard_normal((b, hk, 1, d))).astype(np.float32)
    v = rng.standard_normal((b, hk, skv, dv)).astype(np.float32)
    got = run(ctx, q, k, v, causal)
    want, bound = reference(q, k, v, causal)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.all(np.abs(got[ok] - want[ok]) <= bound[ok])


@pytest.mark.parametrize("d", [64, 80, 128])
def test_masked_and_infinite_entries_stay_where_they_belong(ctx, d):
    """A NaN or infinite value reaches only the queries that see its key; an
    infinite key entry that gives a score of -inf is a key of weight 0."""
    rng = np.random.default_rng(d)
    sq = skv = 75
    q = rng.standard_normal((1, 1, sq, d)).astype(np.float32)
    q[..., 2] = np.abs(q[..., 2]) + 0.1
    k = rng.standard_normal((1, 1, skv, d)).astype(np.float32)
    v = rng.standard_normal((1, 1, skv, d)).astype(np.float32)
    k[0, 0, 5, 2] = -np.inf
    v[0, 0, 70, 3] = np.nan
    v[0, 0, 72, 4] = np.inf
    got = run(ctx, q, k, v, True)[0, 0]
    finite = v.copy()
    finite[0, 0, 70, 3] = finite[0, 0, 72, 4] = 0.0
    assert np.isnan(got[70:, 3]).all() and np.isposinf(got[72:, 4]).all()
    check = np.ones(got.shape, bool)
    check[70:, 3] = check[72:, 4] = False
    assert np.isfinite(got[check]).all()
    for i in range(sq):
        keep = np.delete(np.arange(i + 1), 5) if i >= 5 else np.arange(i + 1)
        x = q[0, 0, i].astype(np.float64)
        s = k[0, 0, keep].astype(np.float64) @ x / np.sqrt(d)
        p = np.exp(s - s.max())
        w = (p @ finite[0, 0, keep].astype(np.float64)) / p.sum()
        lim = (2 * (d / 2 + 4) * EPS * (np.abs(k[0, 0, keep]).astype(np.float64) @ np.abs(x)).max() / np.sqrt(d)
               + 64 * EPS) * np.abs(finite[0, 0, keep]).max()
        assert np.all(np.abs(got[i] - w)[check[i]] <= lim)


@pytest.mark.parametrize("top", [3.0, 300.0, 600.0, 700.0, 1500.0, 3500.0, 4090.0, -700.0, -3500.0, 4100.0, 20000.0])
def test_large_scores_lose_nothing(ctx, top):
    """Scores that are f32 values exactly (one channel, a scale of 1/8), their
    maxima spread over the key tiles and so over the waves, about `top`.

    With the scores exact, a weight is off by the reference's low part (at most
    2^-23 of 1.26, 2.6 eps, eps = 2^-24), the difference's rounding (1 eps) and
    expf (2 eps); both sums of the quotient carry that, 11.2 eps, and the sums
    of 1300 terms in blocks of 32 (f32 roundings of either sign) 5 eps: 16 eps
    of max|v|.  Past 4096 the reference is the max itself and each of a wave's
    at most 6 tiles and the merge scale by an expf (2 eps) with a rounding
    (1 eps), in both sums: 2 x 3 x 7 eps more."""
    rng = np.random.default_rng(int(abs(top)))
    sq, skv, d = 20, 1300, 64
    tile = np.arange(skv) // 32
    s = (top - 0.7 * (tile * 5 % 13) - rng.exponential(1.0, skv)).astype(np.float32)
    q, k = np.zeros((1, 2, sq, d), np.float32), np.zeros((1, 1, skv, d), np.float32)
    q[..., 0], k[0, 0, :, 0] = 8.0, s
    v = rng.choice([-1.0, 1.0], (1, 1, tile[-1] + 1, d)).astype(np.float32)[:, :, tile]  # a tile's weight shows whole
    got = run(ctx, q, k, v, False)
    p = np.exp(s.astype(np.float64) - float(s.max()))
    want = p @ v[0, 0].astype(np.float64) / p.sum()
    assert np.abs(got - want).max() <= (16 if abs(top) < 4096 else 16 + 42) * EPS * np.abs(v).max()


@pytest.mark.parametrize("b,h,hk,sq,skv,d,dv", [
    (26, 16, 4, 1, 38, 64, 64), (26, 16, 4, 16, 128, 64, 64), (26, 16, 4, 16, 127, 64, 64),    # one tile, one, four
    (26, 16, 4, 17, 134, 128, 128), (26, 16, 4, 33, 230, 64, 64), (10, 16, 4, 16, 60, 80, 48),  # two, four, two
])
def test_query_tiles_a_workgroup(ctx, b, h, hk, sq, skv, d, dv):
    """A few queries of many heads: as many query tiles a workgroup as the queries fill."""
    rng = np.random.default_rng(b + sq + skv + d)
    q = rng.standard_normal((b, h, sq, d)).astype(np.float32)
    k = rng.standard_normal((b, hk, skv, d)).astype(np.float32)
    v = rng.standard_normal((b, hk, skv, dv)).astype(np.float32)
    for causal in (False, True):
        want, bound = reference(q, k, v, causal)
        assert np.all(np.abs(run(ctx, q, k, v, causal) - want) <= bound)


@pytest.mark.parametrize("b,h,hk,sq,skv,d,dv", [
    (48, 16, 4, 1, 32, 64, 64), (48, 16, 4, 1, 48, 64, 64), (48, 16, 4, 2, 16, 64, 48),   # a row a workgroup, tiles, a row
    (48, 16, 4, 1, 48, 128, 128), (48, 16, 4, 1, 64, 128, 128), (48, 16, 4, 4, 1, 16, 128),  # a row, tiles, a row
    (20, 16, 4, 1, 8, 64, 64), (20, 16, 4, 1, 9, 64, 64), (16, 16, 4, 4, 8, 16, 16), (16, 16, 4, 4, 9, 16, 16),
])
def test_few_queries_over_few_keys(ctx, b, h, hk, sq, skv, d, dv):
    """Either side of the line between the row kernel and the tiles."""
    rng = np.random.default_rng(b + sq + skv + d)
    q = rng.standard_normal((b, h, sq, d)).astype(np.float32)
    k = rng.standard_normal((b, hk, skv, d)).astype(np.float32)
    v = rng.standard_normal((b, hk, skv, dv)).astype(np.float32)
    for causal in (False, True):
        want, bound = reference(q, k, v, causal)
        got = run(ctx, q, k, v, causal)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ok = ~np.isnan(want)
        assert np.all(np.abs(got - want)[ok] <= bound[ok])
