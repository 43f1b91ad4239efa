"""Decode attention of few sequences on f32 pages (16 waves, one 16-position
tile each and up to four in turn) against the oracle: context lengths around
the edges of a tile, of the 16 waves and of each number of tiles per wave,
every number of heads a workgroup takes, the workgroup counts on both sides of
the choice, page sizes of 4 to 64, NaN behind each context.  The tolerance is
that of the other forms: only the order of the fp32 sums differs."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.test_gpu_attention import build_cache, check, oracle_attention, run_attention

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 33, 63, 255, 256, 257, 272, 273, 511, 512, 513, 768, 769, 1009, 1024, 1025]


def run(hip, n, H, Hkv, hd, ps, ctxs):
    rng = np.random.default_rng(n * H + hd + max(ctxs))
    table, K, V, _ = build_cache(rng, ctxs, Hkv, hd, ps, po.F32, poison=True)
    q = (rng.standard_normal((n, H * hd)) * 2).astype(np.float32)
    got = run_attention(hip, q, table, K, V, ctxs, H, Hkv, hd, ps, po.F32, max(ctxs), repeats=2)
    assert np.array_equal(got[0], got[1])
    check(got[0], oracle_attention(q, table, K, V, ctxs, H, Hkv, hd, ps))


@pytest.mark.parametrize("H,Hkv,hd", [(9, 3, 64), (10, 2, 64), (16, 1, 64), (16, 2, 128), (8, 8, 128)])
@pytest.mark.parametrize("ps", [4, 16, 64])
def test_one_sequence(hip, H, Hkv, hd, ps):
    for c in EDGES:
        if (H // Hkv, hd) == (5, 64) and c <= 256:
            continue  # one sequence of this group: refused
        run(hip, 1, H, Hkv, hd, ps, [c])


@pytest.mark.parametrize("H,Hkv,hd", [(3, 3, 64), (6, 3, 64), (9, 3, 64), (12, 3, 64), (15, 3, 64), (16, 2, 128)])
@pytest.mark.parametrize("n", [15, 29, 43, 85, 86])
@pytest.mark.parametrize("most", [48, 256, 512, 513, 1024])
def test_ragged_batches(hip, H, Hkv, hd, n, most):
    edges = [c for c in EDGES if c <= most][::-1][:n]
    rng = np.random.default_rng(n + most)
    run(hip, n, H, Hkv, hd, 16, edges + rng.integers(1, most + 1, n - len(edges)).tolist())


def test_group_without_a_kernel_stays_refused(hip):
    with pytest.raises(RuntimeError, match="group 5"):
        run(hip, 1, 10, 2, 64, 16, [40])


@pytest.mark.parametrize("how", ["overflow", "infinite"])
@pytest.mark.parametrize("n,H,Hkv,hd,ctx", [
    # n * H <= 256: a workgroup per query head; beyond it (head_dim 64) one per KV head; the matrix cores
    (1, 9, 3, 64, 17), (1, 9, 3, 64, 250), (28, 9, 3, 64, 257), (29, 9, 3, 64, 257), (64, 4, 1, 64, 49),
    (65, 4, 1, 64, 49), (16, 9, 3, 64, 700), (1, 16, 2, 128, 33), (16, 16, 2, 128, 500), (17, 16, 2, 128, 500),
    (86, 9, 3, 64, 200)])
def test_scores_of_minus_infinity(hip, n, H, Hkv, hd, ctx, how):
    """Keys whose score is -inf count as nothing (exp(-inf - max) = 0 in the
    oracle's softmax): the only position of the last tile, a whole tile, and
    single positions, through products that overflow and through an infinite
    key element."""
    ps = 16
    ctxs = [ctx - 16 * (s % 2) if ctx > 32 else ctx for s in range(n)]  # ctx % 16 is the same for all
    rng = np.random.default_rng(n + ctx + hd)
    table, K, V, _ = build_cache(rng, ctxs, Hkv, hd, ps, po.F32, poison=True)
    q = (rng.standard_normal((n, H * hd)) * 2).astype(np.float32)
    q.reshape(n, H, hd)[:, :, 5] = 2 + np.abs(q.reshape(n, H, hd)[:, :, 5])
    low = np.float32(-np.inf if how == "infinite" else -3e38)  # times q > 2: past the range of fp32
    for s, c in enumerate(ctxs):
        last = c - 1 if c % 16 == 1 else c - 3
        for t in [last, 3] + (list(range(16, 32)) if c > 32 else []):
            K[table[s, t // ps], :, t % ps, 5] = low
    got = run_attention(hip, q, table, K, V, ctxs, H, Hkv, hd, ps, po.F32, max(ctxs))
    check(got[0], oracle_attention(q, table, K, V, ctxs, H, Hkv, hd, ps))


@pytest.mark.parametrize("n,H,Hkv,hd,ctx", [(1, 9, 3, 64, 17), (1, 9, 3, 64, 62), (28, 9, 3, 64, 250), (40, 8, 4, 64, 41),
                                            (16, 9, 3, 64, 600), (1, 16, 2, 128, 33), (16, 16, 2, 128, 300)])
def test_infinite_values_stay_infinite(hip, n, H, Hkv, hd, ctx):
    """An infinite element of V makes its output element infinite, as in the
    oracle, also at the position whose row the lanes past the context read."""
    ps = 16
    rng = np.random.default_rng(n + ctx)
    table, K, V, _ = build_cache(rng, [ctx] * n, Hkv, hd, ps, po.F32, poison=True)
    q = rng.standard_normal((n, H * hd)).astype(np.float32)
    first = (ctx - 1) // 16 * 16  # of the last tile
    for s in range(n):
        V[table[s, first // ps], :, first % ps, 7] = np.inf
        V[table[s, 0], :, 1, 9] = -np.inf
    got = run_attention(hip, q, table, K, V, [ctx] * n, H, Hkv, hd, ps, po.F32, ctx)[0]
    want = oracle_attention(q, table, K, V, [ctx] * n, H, Hkv, hd, ps)
    inf = np.isinf(want)
    assert inf.sum() == 2 * n * H and np.array_equal(got[inf], want[inf])
    check(got[~inf], want[~inf])
