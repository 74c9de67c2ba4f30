"""The prefill at head dims up to 128 on the 32-row kernels
(prefill_narrow.hip; MI355X only): shapes at the edges of its row blocks (128
query rows), key tiles (32, two an interval: odd counts leave one key group a
masked tile), key splits and padding, over every cache type, against the
oracle at the prefill's 1e-5 normwise bar.  Every shape is one that the library
sends here (on_32_rows).
"""
import math

import numpy as np
import pytest
import torch

import oracle
from conftest import normwise_err
from gpu_util import dev, host, on_32_rows, pages
from molot_amd import attn
from molot_amd import lib as _lib
from molot_amd.synth import Stream
from test_d512_gpu import caches, on_dev

pytestmark = pytest.mark.gpu

TOL = 1e-5

# (nq, nkv, d, M, N, pos0, window, kind)
SHAPES = [
    (32, 8, 128, 300, 1300, 1000, 0, "f32"),   # splits of odd and even tile counts
    (32, 8, 128, 321, 1055, 734, 0, "bf16"),   # odd rows, N one below a tile's end
    (32, 4, 128, 128, 2400, 2272, 0, "q8"),    # whole row blocks
    (24, 8, 128, 417, 1025, 608, 0, "f32"),    # G = 3: tokens across row blocks
    (64, 64, 64, 129, 2300, 2171, 0, "f32"),   # d = 64, G = 1, one row past a block
    (64, 2, 64, 150, 2000, 1850, 0, "bf16"),
    (64, 2, 64, 150, 2000, 1850, 0, "q8"),
    (32, 8, 128, 700, 700, 0, 0, "bf16"),      # fresh prompt
    (32, 8, 128, 900, 1200, 300, 333, "q8"),   # window cutting tiles at both ends
    (32, 8, 128, 600, 700, 300, 500, "f32"),   # causal end clipped at N
    (32, 8, 96, 400, 1000, 600, 0, "f32"),     # padded to 128
    (32, 8, 100, 400, 1000, 600, 0, "bf16"),   # d % 8 == 4
    (32, 8, 90, 400, 1000, 600, 0, "f32"),     # d % 4 == 2
    (64, 8, 36, 400, 800, 400, 0, "q8"),       # padded Q8, 4-code words
]


def to_cache(kind, K, V, nkv, d):
    if kind == "q8":
        return oracle.q8_cache(K, nkv, d), oracle.q8_cache(V, nkv, d)
    if kind == "bf16":
        return oracle.f32_to_bf16(K), oracle.f32_to_bf16(V)
    return K, V


@pytest.mark.parametrize("shape", SHAPES,
                         ids=[f"{s[0]}q{s[1]}kv_d{s[2]}_M{s[3]}_N{s[4]}_w{s[6]}_{s[7]}"
                              for s in SHAPES])
def test_prefill_narrow_vs_oracle(gpu, shape):
    nq, nkv, d, M, N, pos0, window, kind = shape
    print(f"[case] narrow prefill {shape}", flush=True)
    assert on_32_rows(nq, nkv, d, M, N, window, kind)
    st = Stream(M + N + d + nq + 13)
    Q = st.normal((M, nq, d))
    K, V = caches(st, N, nkv, d, kind)
    O = torch.full((M, nq, d), float("nan"), device="cuda")
    s = 1 / math.sqrt(d)
    attn.attn_prefill_gqa(dev(Q), on_dev(K), on_dev(V), O, nq, nkv, M, N, d, s, pos0, window)
    R = oracle.attn_prefill(Q, K, V, nq, nkv, M, N, d, s, pos0, window)
    err = normwise_err(host(O), R)
    print(f"narrow prefill normwise err {err:.3e}", flush=True)
    assert err < TOL


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
def test_prefill_narrow_row_scales(gpu, d, kind):
    """K and V rows each scaled by their own 2^U(-12, 12), q rows by 2^U(-6, 6),
    and a run of zero V rows: the row units of the scores and of PV, and the
    rows' PV shifts, over scales that move from row to row."""
    print(f"[case] narrow prefill row scales d={d} {kind}", flush=True)
    nq, nkv, M, N, pos0 = 32, 8, 420, 1500, 1080
    rng = np.random.default_rng(177 + len(kind))
    st = Stream(178 + len(kind))
    K, V = (st.normal((N, nkv * d)) * np.exp2(rng.uniform(-12, 12, size=N))[:, None]
            for _ in range(2))
    V[:70] = 0
    Q = (st.normal((M, nq, d)) * np.exp2(rng.uniform(-6, 6, size=(M, nq)))[:, :, None])
    K, V, Q = (x.astype(np.float32) for x in (K, V, Q))
    K, V = to_cache(kind, K, V, nkv, d)
    s = 2.0 ** -12 / math.sqrt(d)
    O = torch.empty((M, nq, d), device="cuda")
    attn.attn_prefill_gqa(dev(Q), on_dev(K), on_dev(V), O, nq, nkv, M, N, d, s, pos0, 0)
    R = oracle.attn_prefill(Q, K, V, nq, nkv, M, N, d, s, pos0, 0)
    err = normwise_err(host(O), R)
    print(f"narrow row scales normwise err {err:.3e}", flush=True)
    assert err < TOL


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kind,n0", [("f32", 0), ("f32", 130), ("bf16", 130), ("q8", 130)])
def test_prefill_narrow_step_pieces(gpu, d, kind, n0):
    """The step's RoPE/append leaves the pieces of its rows (and the zero rows
    after them) where the split kernel would: the attention entry over the same
    cache, which splits every row, gives the step's bits.  A larger prompt
    before it leaves other values in the workspace."""
    print(f"[case] narrow prefill step d={d} {kind} n0={n0}", flush=True)
    nq, nkv, M = 32, 8, 1017 if d == 64 else 601
    st = Stream(190 + d + n0)
    K0, V0 = caches(st, n0 + M, nkv, d, kind)
    q = dev(st.normal((M, nq, d)))
    k, v = (dev(st.normal((M, nkv, d))) for _ in range(2))
    assert on_32_rows(nq, nkv, d, M, n0 + M, 0, kind)
    M2, N2 = M + 300, n0 + M + 900
    Kb, Vb = caches(st, N2, nkv, d, kind, sigma=50.0)
    big = torch.empty((M2, nq, d), device="cuda")
    s = 1 / math.sqrt(d)
    attn.attn_prefill_gqa(dev(st.normal((M2, nq, d))), on_dev(Kb), on_dev(Vb), big, nq, nkv, M2,
                          N2, d, s, N2 - M2, 0)
    Kd, Vd = on_dev(K0), on_dev(V0)
    inv = dev(oracle.rope_inv_freq(500000.0, d))
    O1, O2 = (torch.full((M, nq, d), float("nan"), device="cuda") for _ in range(2))
    attn.prefill_step(q, k, v, Kd, Vd, O1, nq, nkv, d, M, n0, n0, inv, s, 0)
    attn.attn_prefill_gqa(q, Kd, Vd, O2, nq, nkv, M, n0 + M, d, s, n0, 0)
    assert np.isfinite(host(O1)).all()
    assert np.array_equal(host(O1), host(O2))


@pytest.mark.parametrize("nq,nkv,d,M,N", [(32, 8, 128, 300, 1300), (64, 8, 64, 300, 1100)])
@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
def test_prefill_narrow_paged_matches_contiguous(gpu, nq, nkv, d, M, N, kind):
    """Shuffled pages give the bits of the token-major cache: the same pieces
    and the same products."""
    print(f"[case] narrow prefill paged d={d} {kind}", flush=True)
    assert on_32_rows(nq, nkv, d, M, N, 0, kind)
    page = 16
    st = Stream(281 + d)
    Q = dev(st.normal((M, nq, d)))
    K, V = caches(st, N, nkv, d, kind)
    nb = (N + page - 1) // page
    row = st.permutation(nb + 3)[:nb].astype(np.int32)
    Kp, Vp = (on_dev(pages(X, row, nb + 3, nkv, d, page, kind)) for X in (K, V))
    s = 1 / math.sqrt(d)
    Oc, Op = (torch.full((M, nq, d), float("nan"), device="cuda") for _ in range(2))
    attn.attn_prefill_gqa(Q, on_dev(K), on_dev(V), Oc, nq, nkv, M, N, d, s, N - M, 0)
    attn.attn_prefill_paged(Q, Kp, Vp, Op, dev(row), nb, page, nq, nkv, M, N, d, s, N - M, 0)
    assert np.isfinite(host(Oc)).all()
    assert np.array_equal(host(Oc), host(Op))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
def test_prefill_narrow_step_paged_matches_contiguous(gpu, d, kind):
    """The step into a sequence's pages behind 131 cached rows (a page begun): the
    RoPE/append's pieces beside the split of the cached page rows, the bits of
    the step into a token-major cache, and the same rows stored."""
    print(f"[case] narrow prefill step, paged d={d} {kind}", flush=True)
    nq, nkv, M, n0, page = 32, 8, 1017 if d == 64 else 601, 131, 16
    N = n0 + M
    assert on_32_rows(nq, nkv, d, M, N, 0, kind)
    st = Stream(291 + d)
    K, V = caches(st, N, nkv, d, kind)
    q, k, v = (st.normal(x) for x in ((M, nq, d), (M, nkv, d), (M, nkv, d)))
    nb = (N + page - 1) // page
    row = st.permutation(nb + 3)[:nb].astype(np.int32)
    Kc, Vc = on_dev(K), on_dev(V)
    Kp, Vp = (on_dev(pages(X, row, nb + 3, nkv, d, page, kind)) for X in (K, V))
    inv, s = dev(oracle.rope_inv_freq(500000.0, d)), 1 / math.sqrt(d)
    qc, qp = dev(q), dev(q)
    Oc, Op = (torch.full((M, nq, d), float("nan"), device="cuda") for _ in range(2))
    attn.prefill_step(qc, dev(k), dev(v), Kc, Vc, Oc, nq, nkv, d, M, n0, n0, inv, s, 0)
    attn.prefill_step_paged(qp, dev(k), dev(v), Kp, Vp, Op, dev(row), nb, page, nq, nkv, d, M, n0,
                            n0, inv, s, 0)
    assert np.isfinite(host(Oc)).all()
    assert np.array_equal(host(Oc), host(Op)) and np.array_equal(host(qc), host(qp))
    bits = lambda t: host(t.view(torch.int16) if kind == "bf16" else t)  # noqa: E731
    for c, p in ((Kc, Kp), (Vc, Vp)):
        want = pages(bits(c), row, nb + 3, nkv, d, page, kind)
        got = bits(p).reshape(want.shape)
        assert np.array_equal(got[row], want[row])


@pytest.mark.parametrize("nq,nkv,d,M,N,kind", [
    (16, 16, 128, 100, 7000, "bf16"),  # one row block a head, which 16 key splits multiply to the CUs
    (16, 16, 128, 100, 7000, "q8"),
    (32, 8, 128, 64, 8000, "f32"),     # two
    (32, 8, 128, 128, 4100, "bf16"),   # four, over too few keys
    (8, 2, 512, 2, 30000, "q8"),       # a few rows over a long cache
    (8, 2, 512, 7, 8000, "f32"),
])
def test_prompts_that_keep_the_smaller_ones_path(gpu, nq, nkv, d, M, N, kind):
    """Work enough for the 32-row kernels, but too few rows to pay for the split of
    the cached rows: the bits of the path without a workspace."""
    print(f"[case] few rows {nq}/{nkv}/{d} M={M} N={N} {kind}", flush=True)
    assert M * nq * N >= 400000 if d > 256 else M * nq * N * d >= 1200000000
    assert not on_32_rows(nq, nkv, d, M, N, 0, kind)
    st = Stream(311 + M)
    Q = dev(st.normal((M, nq, d)))
    K, V = (on_dev(x) for x in caches(st, N, nkv, d, kind))
    out = []
    _lib.load().molot_hip_set_block_order(0)  # the vector-ALU kernel: the same sums every time
    try:
        for on in (True, False):
            attn.set_prefill_presplit(on)
            O = torch.full((M, nq, d), float("nan"), device="cuda")
            attn.attn_prefill_gqa(Q, K, V, O, nq, nkv, M, N, d, 1 / math.sqrt(d), N - M, 0)
            out.append(host(O))
    finally:
        attn.set_prefill_presplit(True)
        _lib.load().molot_hip_set_block_order(1)
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])
