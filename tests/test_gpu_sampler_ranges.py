"""Device sampler at the edges of its sub-range maxima path, against
Sampler::sample (sampler.cpp:57-128) restated in numpy float32: the sorted
candidates by (p descending, index ascending), exp(p - max), the sequential
sums in order, top-p, and the cumulative sum against the uniform.  A uniform
that lands within 1e-5 of a cumulative boundary is moved to the middle of its
interval (device expf against numpy's differs in the last place)."""
import numpy as np
import pytest

from tests.test_gpu_sampler import device_sample

pytestmark = pytest.mark.gpu


def candidates(l, T, k, top_p):
    p = (l / np.float32(T)).astype(np.float32)
    o = np.lexsort((np.arange(l.size), -p))[:k]
    e = np.exp(p[o] - p[o[0]]).astype(np.float32)
    e = (e / np.cumsum(e, dtype=np.float32)[-1]).astype(np.float32)
    if 0.0 < top_p < 1.0:
        cs = np.cumsum(e, dtype=np.float32)
        m = int(np.argmax(cs >= np.float32(top_p))) + 1 if (cs >= np.float32(top_p)).any() else k
        o, e = o[:m], (e[:m] / cs[m - 1]).astype(np.float32)
    return o, np.cumsum(e, dtype=np.float32)


def pick(o, cs, r):
    hit = np.nonzero(np.float32(r) <= cs)[0]
    return o[hit[0]] if hit.size else o[-1]


@pytest.mark.parametrize("V", [16380, 16448, 16452, 20004, 151936])
@pytest.mark.parametrize("k", [1, 40, 64, 65, 512, 513])
def test_sampling_with_sub_range_maxima(hip, V, k):
    rng = np.random.default_rng(V + k)
    rows = []
    q = (V // 4 + 3) // 4  # float4s of a sub-range
    for kind in range(6):
        l = (rng.standard_normal(V) * 2).astype(np.float32)
        if kind == 1:  # the row's largest values at the sub-ranges' ends
            for s in range(1, 5):
                l[min(V, 4 * q * s) - 4:min(V, 4 * q * s)] = 20 + rng.random(4)
        elif kind == 2:  # many equal values around the cutoff
            l = np.round(l * 4) / 4
        elif kind == 3:  # the candidates all in one thread's reach
            l[4 * np.arange(8) * 1024 % (V - 4)] = 15 + np.arange(8)
        elif kind == 4:  # a masked row (left to the search over the row)
            l[::3] = -np.inf
        elif kind == 5:  # distinct logits that round to one p
            l[100:100 + 64] = np.nextafter(np.float32(9), np.float32(10)) + np.float32(1e-6) * np.arange(64)
        rows.append(l.astype(np.float32))
    L = np.stack(rows)
    for T, top_p in ((0.8, 0.9), (1.7, 1.0), (3.0, 0.5)):
        want, uni = [], []
        for l in rows:
            o, cs = candidates(l, T, k, top_p)
            r = np.float32(rng.random())
            j = int(np.searchsorted(cs, r))
            if np.abs(cs - r).min() < 1e-5:
                lo = cs[j - 1] if j > 0 else np.float32(0)
                r = np.float32((float(lo) + float(cs[min(j, cs.size - 1)])) / 2)
            clear = np.abs(cs - r).min() >= 1e-6  # else several boundaries in one place: any of their tokens
            want.append(pick(o, cs, r) if clear else None)
            uni.append(r)
        got, _ = device_sample(hip, L, (T, k, top_p, 1.0), uniforms=np.array(uni, np.float32))
        for kind, (g, w) in enumerate(zip(got, want)):
            assert w is None or g == w, f"V={V} k={k} T={T} top_p={top_p} kind={kind}: {g} against {w}"


@pytest.mark.parametrize("V", [16448, 40000, 151936])
@pytest.mark.parametrize("k", [1, 40, 100, 512])
def test_rows_left_to_the_search(hip, V, k):
    """Rows whose sub-range maxima are not finite or whose bound more than 4,096
    values reach go to the search, or to the radix select, with what the first
    read of the row found."""
    rng = np.random.default_rng(V * k)
    base = (rng.standard_normal(V) * 2).astype(np.float32)
    rows = [base.copy() for _ in range(9)]
    rows[0][V // 2:] = -np.inf          # a constrained vocabulary
    rows[1][700:] = -np.inf
    rows[2][5:4105] = -np.inf           # a sub-range of some threads only
    rows[3] = np.minimum(base, 2.0)     # a sixth of the row equal, at the top
    rows[4][:] = 1.5
    rows[5] = np.where(rng.random(V) < 0.3, 5.0, -1.0)
    rows[6][:5000] += 20                # more than 4,096 above the rest, all distinct
    rows[7] = np.round(base * 2) / 2
    rows[8][11] = np.inf                # its p - max is NaN: the last candidate
    rows = [r.astype(np.float32) for r in rows]
    for T, top_p in ((0.8, 0.9), (2.0, 1.0)):
        want, uni = [], []
        for i, l in enumerate(rows):
            with np.errstate(invalid="ignore"):
                o, cs = candidates(l, T, k, top_p)
            r = np.float32(rng.random())
            if not np.isfinite(cs).all():
                want.append(o[-1])
            else:
                j = min(int(np.searchsorted(cs, r)), cs.size - 1)
                if np.abs(cs - r).min() < 1e-5:
                    r = np.float32(((float(cs[j - 1]) if j else 0.0) + float(cs[j])) / 2)
                want.append(pick(o, cs, r) if np.abs(cs - r).min() >= 1e-6 else None)
            uni.append(r)
        got, _ = device_sample(hip, np.stack(rows), (T, k, top_p, 1.0), uniforms=np.array(uni, np.float32))
        for i, (g, w) in enumerate(zip(got, want)):
            assert w is None or g == w, f"V={V} k={k} T={T} row {i}: {g} against {w}"


@pytest.mark.parametrize("V", [16448, 151936])
@pytest.mark.parametrize("k", [1, 40, 100])
def test_temperatures_that_overflow(hip, V, k):
    """logit / T past the range of fp32: every such p is the same infinity, the
    candidates are those of the lowest index, their exponentials NaN, and the
    token the last candidate (no sum reaches top_p or the uniform)."""
    rng = np.random.default_rng(V + k)
    L = (rng.standard_normal((5, V)) * 2).astype(np.float32)
    L[1] -= 1000  # every p is -inf
    L[2] = np.round(L[2])
    L[3, : V // 2] -= 50
    L[4] *= np.float32(1e3)
    for top_p in (0.9, 1.0):
        with np.errstate(over="ignore", invalid="ignore"):
            want = [candidates(l, 1e-38, k, top_p)[0][-1] for l in L]
        got, _ = device_sample(hip, L, (1e-38, k, top_p, 1.0), uniforms=np.full(5, 0.5, np.float32))
        assert list(got) == want, f"V={V} k={k} top_p={top_p}"
