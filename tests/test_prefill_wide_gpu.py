"""The prefill at head dims above 256 on the matrix cores (prefill_wide.hip;
MI355X only): shapes at the edges of its row blocks (64 query rows), key tiles
(32), key splits and padding to D = 512, over every cache type, against the
oracle at the prefill's 1e-5 normwise bar.  Every shape is one that the library
sends here (on_32_rows).
"""
import math

import numpy as np
import pytest
import torch

import oracle
from conftest import normwise_err
from gpu_util import dev, host, on_32_rows
from molot_amd import attn
from molot_amd.synth import Stream
from test_d512_gpu import caches, on_dev

pytestmark = pytest.mark.gpu

TOL = 1e-5

# (nq, nkv, d, M, N, pos0, window, kind)
SHAPES = [
    (8, 8, 512, 64, 1000, 936, 0, "f32"),      # G = 1: one full row block a head
    (8, 8, 512, 65, 1001, 936, 0, "bf16"),     # one row past it, odd N
    (8, 2, 512, 250, 250, 0, 0, "f32"),        # fresh prompt, blocks of 16 tokens and a remainder
    (6, 2, 512, 333, 333, 0, 0, "q8"),         # G = 3: tokens across row blocks
    (16, 1, 512, 9, 4000, 3991, 0, "f32"),     # few rows, many key splits (combine_kernel)
    (8, 2, 512, 90, 1500, 1410, 700, "bf16"),  # window cutting tiles at both ends
    (16, 2, 512, 800, 900, 300, 33, "f32"),    # window of two tiles, causal end clipped at N
    (32, 2, 300, 40, 500, 460, 0, "f32"),      # padded: d % 8 == 4
    (16, 2, 510, 60, 500, 440, 0, "f32"),      # d % 4 == 2: two-element loads and stores
    (16, 2, 258, 60, 500, 440, 0, "bf16"),
    (32, 2, 420, 130, 560, 430, 100, "q8"),    # padded Q8, 4-code words
]


@pytest.mark.parametrize("shape", SHAPES,
                         ids=[f"{s[0]}q{s[1]}kv_d{s[2]}_M{s[3]}_N{s[4]}_w{s[6]}_{s[7]}"
                              for s in SHAPES])
def test_prefill_wide_vs_oracle(gpu, shape):
    nq, nkv, d, M, N, pos0, window, kind = shape
    print(f"[case] wide prefill {shape}", flush=True)
    assert on_32_rows(nq, nkv, d, M, N, window, kind)
    st = Stream(M + N + d + nq + 11)
    Q = st.normal((M, nq, d))
    K, V = caches(st, N, nkv, d, kind)
    O = torch.full((M, nq, d), float("nan"), device="cuda")
    s = 1 / math.sqrt(d)
    attn.attn_prefill_gqa(dev(Q), on_dev(K), on_dev(V), O, nq, nkv, M, N, d, s, pos0, window)
    R = oracle.attn_prefill(Q, K, V, nq, nkv, M, N, d, s, pos0, window)
    err = normwise_err(host(O), R)
    print(f"wide prefill normwise err {err:.3e}", flush=True)
    assert err < TOL


@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
def test_prefill_wide_row_scales(gpu, kind):
    """K and V rows each scaled by their own 2^U(-12, 12), q rows by
    2^U(-6, 6): the units of the scores and of PV, and the rows' PV shifts
    (taken kRoom bits low), over scales that move from row to row."""
    print(f"[case] wide prefill row scales {kind}", flush=True)
    nq, nkv, d, M, N, pos0 = 8, 2, 512, 90, 650, 560
    rng = np.random.default_rng(77 + len(kind))
    st = Stream(78 + len(kind))
    K, V = (st.normal((N, nkv * d)) * np.exp2(rng.uniform(-12, 12, size=N))[:, None]
            for _ in range(2))
    Q = (st.normal((M, nq, d)) * np.exp2(rng.uniform(-6, 6, size=(M, nq)))[:, :, None])
    K, V, Q = (x.astype(np.float32) for x in (K, V, Q))
    if kind == "q8":
        K, V = oracle.q8_cache(K, nkv, d), oracle.q8_cache(V, nkv, d)
    elif kind == "bf16":
        K, V = oracle.f32_to_bf16(K), oracle.f32_to_bf16(V)
    s = 2.0 ** -12 / math.sqrt(d)
    O = torch.empty((M, nq, d), device="cuda")
    attn.attn_prefill_gqa(dev(Q), on_dev(K), on_dev(V), O, nq, nkv, M, N, d, s, pos0, 0)
    R = oracle.attn_prefill(Q, K, V, nq, nkv, M, N, d, s, pos0, 0)
    err = normwise_err(host(O), R)
    print(f"wide row scales normwise err {err:.3e}", flush=True)
    assert err < TOL


@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
def test_prefill_wide_paged_matches_contiguous(gpu, kind):
    """Shuffled pages give the bits of the token-major cache: the same pieces
    and the same products."""
    print(f"[case] wide prefill paged {kind}", flush=True)
    nq, nkv, d, M, N, page = 8, 2, 512, 120, 520, 16
    st = Stream(81)
    Q = dev(st.normal((M, nq, d)))
    K, V = caches(st, N, nkv, d, kind)
    nb = (N + page - 1) // page
    row = st.permutation(nb + 3)[:nb].astype(np.int32)
    pools = []
    for X in (K, V):
        if kind == "q8":
            P = np.zeros((nb + 3, oracle.q8_block_bytes(nkv, d, page)), np.uint8)
            codes = P[:, :nkv * page * d].reshape(nb + 3, nkv, page, d)
            scales = P[:, nkv * page * d:].reshape(nb + 3, -1, 4)
            for t in range(N):
                codes[row[t // page], :, t % page] = X[t, :nkv * d].reshape(nkv, d)
                sc = X[t, nkv * d:nkv * d + 4 * nkv].reshape(nkv, 4)
                for h in range(nkv):
                    scales[row[t // page], h * page + t % page] = sc[h]
        else:
            P = np.zeros((nb + 3, nkv, page, d), X.dtype)
            for t in range(N):
                P[row[t // page], :, t % page] = X[t].reshape(nkv, d)
        pools.append(on_dev(P.reshape(nb + 3, -1)))
    s = 1 / math.sqrt(d)
    Oc, Op = (torch.full((M, nq, d), float("nan"), device="cuda") for _ in range(2))
    attn.attn_prefill_gqa(Q, on_dev(K), on_dev(V), Oc, nq, nkv, M, N, d, s, N - M, 0)
    attn.attn_prefill_paged(Q, pools[0], pools[1], Op, dev(row), nb, page, nq, nkv, M, N, d, s,
                            N - M, 0)
    assert np.isfinite(host(Oc)).all()
    assert np.array_equal(host(Oc), host(Op))
