"""Workgroups that hold a whole context of 257 to 1,024 positions (8, 12 and
16 waves) against the oracle, on both sides of every length and workgroup
count where the automatic choice changes, with NaN (fp16, f32) behind each
context.  Tolerances are those of the chunk and split forms' tests: the
arithmetic per tile is the same, only the order of the fp32 sums differs."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.test_gpu_attention import build_cache, check, oracle_attention, run_attention
from tests.test_gpu_kv_int8 import build_i8_cache, oracle_i8, run_i8
from tests.test_gpu_kv_int8 import check as check_i8

pytestmark = pytest.mark.gpu

# (sequences, KV heads, query heads per KV head, head_dim, longest context): n * Hkv in
# 129..256 takes 12 waves up to 768 positions, 193..256 takes 16 up to 1,024
SHAPES = [(3, 2, 8, 128, 257), (5, 3, 3, 64, 512), (2, 1, 16, 128, 500), (33, 4, 2, 64, 513), (32, 8, 16, 128, 768),
          (43, 3, 1, 64, 700), (43, 6, 1, 64, 768), (25, 8, 16, 128, 1024), (49, 4, 2, 64, 1000), (64, 4, 3, 64, 769),
          (48, 4, 2, 64, 1024), (65, 4, 2, 64, 1024), (50, 4, 2, 64, 1025)]


def lengths(rng, n, most):
    edges = [most, 1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 639, 640, 767, 768, 769, 960, 961]
    edges = [c for c in edges if c <= most][:n]
    return edges + rng.integers(1, most + 1, n - len(edges)).tolist()


@pytest.mark.parametrize("n,Hkv,G,hd,most", SHAPES)
@pytest.mark.parametrize("kv_dtype", [po.F16, po.F32])
@pytest.mark.parametrize("ps", [4, 16])
def test_attention_whole_context_workgroups(hip, n, Hkv, G, hd, most, kv_dtype, ps):
    rng = np.random.default_rng(n * most + hd)
    ctxs = lengths(rng, n, most)
    table, K, V, _ = build_cache(rng, ctxs, Hkv, hd, ps, kv_dtype, poison=True)
    q = (rng.standard_normal((n, Hkv * G * hd)) * 2).astype(np.float32)
    got = run_attention(hip, q, table, K, V, ctxs, Hkv * G, Hkv, hd, ps, kv_dtype, most, repeats=2)
    assert np.array_equal(got[0], got[1])
    check(got[0], oracle_attention(q, table, K, V, ctxs, Hkv * G, Hkv, hd, ps))


@pytest.mark.parametrize("n,Hkv,G,hd,most", SHAPES)
def test_attention_i8_whole_context_workgroups(hip, n, Hkv, G, hd, most):
    rng = np.random.default_rng(n * most + hd + 1)
    ctxs = lengths(rng, n, most)
    table, K8, Ks, V8, Vs, _ = build_i8_cache(rng, ctxs, Hkv, hd, 16)
    q = rng.standard_normal((n, Hkv * G * hd)).astype(np.float32)
    got = run_i8(hip, q, table, K8, Ks, V8, Vs, ctxs, Hkv * G, Hkv, hd, 16)
    check_i8(got[0], oracle_i8(q, table, K8, Ks, V8, Vs, ctxs, Hkv * G, Hkv, hd, 16))
