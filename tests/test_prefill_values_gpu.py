"""The 32-row prefill kernels (prefill_narrow.hip, prefill_wide.hip; MI355X only)
over values at the ends of the number range: subnormal query rows, keys without
a V value yet before tiny ones; against the oracle at the prefill's 1e-5
normwise bar.  Every shape has the work from which the library takes these
kernels.
"""
import math

import numpy as np
import pytest
import torch

import oracle
from conftest import normwise_err
from gpu_util import dev, host
from molot_amd import attn
from molot_amd.synth import Stream
from test_d512_gpu import caches, on_dev
from test_prefill_narrow_gpu import to_cache

pytestmark = pytest.mark.gpu

TOL = 1e-5

# (nq, nkv, d, M, N): the last M of N positions
NARROW = (32, 8, 128, 300, 1300)
WIDE = (8, 2, 512, 150, 700)


def run(Q, K, V, nq, nkv, d, window=0):
    """(kernel, oracle) outputs of a prompt at the end of its cache."""
    M, N, s = Q.shape[0], K.shape[0], 1 / math.sqrt(d)
    assert M * nq * N >= 400000 if d > 256 else M * nq * N * (64 if d <= 64 else 128) >= 1.2e9
    O = torch.full((M, nq, d), -77.0, device="cuda")
    attn.attn_prefill_gqa(dev(Q), on_dev(K), on_dev(V), O, nq, nkv, M, N, d, s, N - M, window)
    return host(O), oracle.attn_prefill(Q, K, V, nq, nkv, M, N, d, s, N - M, window)


@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
@pytest.mark.parametrize("shape", [NARROW, WIDE], ids=["narrow", "wide"])
def test_subnormal_query_rows(gpu, shape, kind):
    """Every fourth query row of magnitude 1e-42, the others ordinary: its scores
    are zero, those of its masked keys still minus infinity."""
    nq, nkv, d, M, N = shape
    print(f"[case] subnormal q {shape} {kind}", flush=True)
    st = Stream(701 + d)
    Q = st.normal((M, nq, d))
    Q[::4] *= np.float32(1e-42)
    assert (Q[::4] != 0).any()
    K, V = caches(st, N, nkv, d, kind)
    O, R = run(Q, K, V, nq, nkv, d)
    assert np.isfinite(O).all()
    assert normwise_err(O, R) < TOL
    assert normwise_err(O[::4], R[::4]) < TOL


@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
@pytest.mark.parametrize("shape", [NARROW, WIDE], ids=["narrow", "wide"])
def test_tiny_values_after_zero_ones(gpu, shape, kind):
    """V zero over the first tiles and of magnitude 1e-32 after them: the first
    V unit a row meets is taken however small it is."""
    nq, nkv, d, M, N = shape
    print(f"[case] tiny V after zeros {shape} {kind}", flush=True)
    st = Stream(711 + d)
    Q, K, V = st.normal((M, nq, d)), st.normal((N, nkv * d)), st.normal((N, nkv * d))
    V[:200] = 0
    V[200:] *= np.float32(1e-32)
    K, V = to_cache(kind, K, V, nkv, d)
    O, R = run(Q, K, V, nq, nkv, d)
    assert np.abs(R).max() > 1e-34
    assert normwise_err(O, R) < TOL
