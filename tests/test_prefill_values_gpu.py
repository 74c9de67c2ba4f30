"""The 32-row prefill kernels (prefill_narrow.hip, prefill_wide.hip; MI355X only)
over values at the ends of the number range: subnormal query rows, keys without
a V value yet before tiny ones, rows that are not finite; against the oracle at the prefill's 1e-5
normwise bar.  Every shape has the work from which the library takes these
kernels.
"""
import math

import numpy as np
import pytest
import torch

import oracle
from conftest import normwise_err
from gpu_util import dev, host, on_32_rows, pages
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
    kind = {np.dtype(np.uint8): "q8", np.dtype(np.uint16): "bf16"}.get(K.dtype, "f32")
    assert on_32_rows(nq, nkv, d, M, N, window, kind)
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


OWN = [
    # (nq, nkv, d, M, N, window, kind): head dims at which each query row reads its own keys
    (8, 2, 512, 150, 700, 0, "f32"),
    (8, 2, 512, 150, 700, 0, "bf16"),
    (6, 2, 512, 200, 500, 0, "q8"),
    (16, 2, 300, 150, 600, 0, "f32"),
    (8, 2, 512, 300, 900, 200, "f32"),     # rows that have the marked keys behind their window
    (16, 1, 512, 9, 4000, 0, "f32"),       # key splits
    (32, 8, 100, 400, 1000, 0, "f32"),
    (32, 8, 90, 500, 900, 0, "bf16"),
    (64, 8, 36, 500, 800, 0, "q8"),
    (32, 8, 100, 300, 1300, 0, "f32"),     # key splits
]


def spoil(K, V, nkv, d, kind, M):
    """An infinite and a NaN value of V, and (not Q8) a K element of minus
    infinity, in three of the prompt's own rows."""
    N = K.shape[0]
    t1, t2, t3 = N - M + M // 3, N - M + M // 2, N - M + 2 * M // 3
    for h in range(nkv):
        if kind == "q8":
            V[t1, nkv * d + 4 * h:][:4] = np.frombuffer(np.float32(np.inf).tobytes(), np.uint8)
            V[t2, nkv * d + 4 * h:][:4] = np.frombuffer(np.float32(np.nan).tobytes(), np.uint8)
        else:
            bits = (lambda x: x) if kind == "f32" else \
                (lambda x: int(oracle.f32_to_bf16(np.asarray([x], np.float32))[0]))
            V[t1, h * d + 3] = bits(np.inf)
            V[t2, h * d + d - 1] = bits(np.nan)
            K[t3, h * d] = bits(-np.inf)


def same(O, R):
    """The same values that are not finite, and the others to the parity bar."""
    assert np.array_equal(np.isnan(O), np.isnan(R))
    inf = np.isinf(R)
    assert np.array_equal(np.isinf(O), inf) and np.array_equal(O[inf], R[inf])
    fin = np.isfinite(R)
    assert 0 < fin.sum() < R.size
    assert normwise_err(O[fin], R[fin]) < TOL


@pytest.mark.parametrize("case", OWN, ids=[f"{c[0]}q{c[1]}kv_d{c[2]}_M{c[3]}_N{c[4]}_w{c[5]}_{c[6]}"
                                           for c in OWN])
def test_non_finite_rows_reach_their_queries_alone(gpu, case):
    nq, nkv, d, M, N, window, kind = case
    print(f"[case] non-finite rows {case}", flush=True)
    st = Stream(721 + d + N)
    Q = st.normal((M, nq, d))
    Q[:, :, 0] = np.abs(Q[:, :, 0]) + 0.1
    K, V = caches(st, N, nkv, d, kind)
    spoil(K, V, nkv, d, kind, M)
    O, R = run(Q, K, V, nq, nkv, d, window)
    same(O, R)


@pytest.mark.parametrize("d", [100, 512])
def test_rows_out_of_the_pieces_range(gpu, d):
    """Finite rows whose scaled pieces would overflow a score (K of 1e30 under q
    of 1e-30) or keep fewer bits (V of 1e-35 beside ordinary rows whose weight
    is next to nothing)."""
    nq, nkv, M, N = (8, 2, 150, 700) if d == 512 else (32, 8, 400, 1000)
    print(f"[case] rows out of the pieces' range d={d}", flush=True)
    st = Stream(741 + d)
    Q, K, V = st.normal((M, nq, d)), st.normal((N, nkv * d)), st.normal((N, nkv * d))
    O, R = run(Q * np.float32(1e-35), K * np.float32(1e35), V, nq, nkv, d)
    assert normwise_err(O, R) < TOL
    O, R = run(Q, K, V * np.float32(1e-35), nq, nkv, d)
    assert normwise_err(O, R) < TOL


@pytest.mark.parametrize("kind", ["f32", "q8"])
def test_non_finite_rows_paged(gpu, kind):
    """The same through shuffled pages."""
    print(f"[case] non-finite rows, paged {kind}", flush=True)
    nq, nkv, d, M, N, page = 8, 2, 512, 150, 700, 16
    st = Stream(731)
    Q = st.normal((M, nq, d))
    Q[:, :, 0] = np.abs(Q[:, :, 0]) + 0.1
    K, V = caches(st, N, nkv, d, kind)
    spoil(K, V, nkv, d, kind, M)
    nb = (N + page - 1) // page
    row = st.permutation(nb + 3)[:nb].astype(np.int32)
    pools = [on_dev(pages(X, row, nb + 3, nkv, d, page, kind)) for X in (K, V)]
    s = 1 / math.sqrt(d)
    O = torch.full((M, nq, d), -77.0, device="cuda")
    attn.attn_prefill_paged(dev(Q), pools[0], pools[1], O, dev(row), nb, page, nq, nkv, M, N, d, s,
                            N - M, 0)
    same(host(O), oracle.attn_prefill(Q, K, V, nq, nkv, M, N, d, s, N - M, 0))
