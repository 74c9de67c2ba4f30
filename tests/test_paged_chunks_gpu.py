"""Paged batches on the matrix-core kernel whose chunks follow the sequences'
lengths (paged_chunk; MI355X only): batches on both sides of each line of
dyn_chunk, more sequences than a wave has lanes, single rows beside long
contexts, windows, explicit positions, empty sequences; against the oracle, and
against the same launch with chunks forced from the host.
"""
import ctypes
import math

import numpy as np
import pytest
import torch

import oracle
from conftest import normwise_err
from gpu_util import dev, dev_bf16, host, make_paged, oracle_paged
from molot_amd import attn
from molot_amd import lib as _lib
from molot_amd.synth import Stream, f32_to_bf16

pytestmark = pytest.mark.gpu

TOL = 1e-5
PAGE = 16


def batch(lens, nq, nkv, d, seed):
    """make_paged's problem with the given rows (new token included) a sequence."""
    P = make_paged(len(lens), nq, nkv, d, 1, 2, seed=seed)
    n = np.asarray(lens, np.int32)
    blocks = (n + PAGE - 1) // PAGE
    st = Stream(seed + 1)
    nblk = int(blocks.sum()) + 5
    perm = st.permutation(nblk)
    bt = np.zeros((len(lens), max(1, int(blocks.max()))), np.int32)
    at = 0
    for b, k in enumerate(blocks):
        bt[b, :k] = perm[at:at + k]
        at += k
    P.update(n=n, bt=bt, max_blocks=bt.shape[1],
             Kp=f32_to_bf16(st.normal((nblk, nkv, PAGE, d))),
             Vp=f32_to_bf16(st.normal((nblk, nkv, PAGE, d))))
    return P


CASES = [
    # (name, lens, nq, nkv, d, window)
    ("one row", [1], 32, 8, 128, 0),
    ("one long", [9000], 32, 8, 128, 0),                       # one round, 256-row chunks
    ("edges of 128", [127, 128, 129, 255, 256, 257, 1], 32, 8, 128, 0),
    ("uneven", [1, 2999, 37, 800, 1500, 5, 2100, 640, 300, 1200, 90, 2500, 33], 32, 8, 128, 0),
    ("64 short", [40 + 13 * i for i in range(64)], 32, 8, 128, 0),  # one chunk each
    ("64 long", [700 + 30 * i for i in range(64)], 32, 8, 64, 0),   # kDynRound rows
    ("130 sequences", [1 + (37 * i) % 400 for i in range(130)], 16, 4, 64, 0),
    ("window", [3000, 10, 1025, 1024, 5000], 64, 8, 128, 1024),
    ("G = 1, many heads", [900, 20, 333], 40, 40, 64, 0),
    # one row either side of where a chunk grows by 128 rows: the step attends
    # one cached row less than its longest sequence counts
    ("one of 8065", [8065], 32, 8, 128, 0),
    ("one of 16129", [16129], 32, 8, 64, 0),
    ("one of 1511, 40 heads", [1511], 40, 40, 64, 0),
    ("one long of four", [7681, 1, 1, 1], 32, 8, 128, 0),
    ("one long of 13", [6529] + 12 * [1], 32, 8, 128, 0),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0].replace(" ", "_") for c in CASES])
def test_paged_step_vs_oracle(gpu, case):
    name, lens, nq, nkv, d, window = case
    print(f"[case] paged chunks: {name}", flush=True)
    P = batch(lens, nq, nkv, d, 300 + len(lens))
    B = len(lens)
    inv = oracle.rope_inv_freq(500000.0, d)
    s = 1 / math.sqrt(d)
    q, K, V = dev(P["q"]), dev_bf16(P["Kp"]), dev_bf16(P["Vp"])
    O = torch.full((B, nq, d), float("nan"), device="cuda")
    attn.decode_step_paged(q, dev(P["k_new"]), dev(P["v_new"]), K, V, O, dev(P["bt"].reshape(-1)),
                           dev(P["n"]), None, B, P["max_blocks"], nq, nkv, d, PAGE, dev(inv), s,
                           window)
    q_ref, _, _, _ = oracle_paged(P, inv, s, window)
    np.testing.assert_allclose(host(q), q_ref, rtol=2e-6, atol=4e-6)
    # attention on the GPU's own pages
    Kh, Vh = (host(x.view(torch.int16)).view(np.uint16) for x in (K, V))
    R = oracle.attn_decode_paged(host(q), Kh, Vh, P["bt"], P["n"], None, B, P["max_blocks"], nq,
                                 nkv, d, PAGE, s, window)
    for b in range(B):
        assert normwise_err(host(O[b]), R[b]) < TOL, (b, lens[b])


@pytest.mark.parametrize("lens", [[4097], [8064], [6570, 200, 300, 107], [33, 700, 5]])
@pytest.mark.parametrize("bound", ["5/4", "table"])
def test_paged_step_loose_max_seq_len(gpu, lens, bound):
    """max_seq_len as a bound above the longest sequence (a captured graph's, a
    table's capacity) gives the result of the exact one."""
    print(f"[case] paged chunks, loose bound: {lens} {bound}", flush=True)
    nq, nkv, d = 32, 8, 128
    P = batch(lens, nq, nkv, d, 500 + len(lens))
    B, width = len(lens), 2048  # 32768 rows a sequence
    table = np.zeros((B, width), np.int32)
    table[:, :P["max_blocks"]] = P["bt"]
    inv, s = oracle.rope_inv_freq(500000.0, d), 1 / math.sqrt(d)
    q, K, V = dev(P["q"]), dev_bf16(P["Kp"]), dev_bf16(P["Vp"])
    kn, vn, bt, n, iv = (dev(x) for x in (P["k_new"], P["v_new"], table, P["n"], inv))
    O = torch.full((B, nq, d), float("nan"), device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    most = width * PAGE if bound == "table" else max(lens) * 5 // 4
    status = _lib.load().molot_hip_decode_step_paged(
        p(q), p(kn), p(vn), p(K), p(V), p(O), p(bt), p(n), None, B, width, most, nq, nkv, d, PAGE,
        p(iv), s, 0, attn.KV_BF16, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert status == 0
    Kh, Vh = (host(x.view(torch.int16)).view(np.uint16) for x in (K, V))
    R = oracle.attn_decode_paged(host(q), Kh, Vh, table, P["n"], None, B, width, nq, nkv, d, PAGE,
                                 s, 0)
    for b in range(B):
        assert normwise_err(host(O[b]), R[b]) < TOL, (b, lens[b])


def pools(P, nkv, d, kind, seed):
    """P's K and V pools on the device, or Q8 ones of as many blocks."""
    if kind == "bf16":
        return dev_bf16(P["Kp"]), dev_bf16(P["Vp"])
    st = Stream(seed)
    nblk, out = P["Kp"].shape[0], []
    for _ in range(2):
        X = np.zeros((nblk, oracle.q8_block_bytes(nkv, d, PAGE)), np.uint8)
        cut = nkv * PAGE * d
        codes = np.clip(np.rint(st.normal((nblk, cut)) * 32), -127, 127).astype(np.int8)
        X[:, :cut] = codes.view(np.uint8)
        sc = (np.abs(st.normal((nblk, nkv * PAGE))) * 0.03 + 0.01).astype(np.float32)
        X[:, cut:cut + 4 * nkv * PAGE] = sc.view(np.uint8)
        out.append(dev(X))
    return out


@pytest.mark.parametrize("kind", ["bf16", "q8"])
@pytest.mark.parametrize("lens, nq, nkv, d", [
    # the others leave the chunks short: the long ones may have more of them than a
    # batch of long ones would (dyn_plan's likely), in the combine's first round
    # of loads (9 to 32, 33 to 64, 65 to 128 chunks) and past it
    ([1100] + 40 * [10], 16, 2, 128),
    ([6000] + 40 * [10], 16, 2, 128),
    ([12000, 9000] + 20 * [10], 16, 2, 128),
    ([14000] + 40 * [10], 8, 1, 64),
    # several rounds: 768 rows a chunk, Q8 768, 1024 or 1536
    ([1025, 1024, 4097, 4096] + 60 * [1030], 32, 8, 64),
    ([2049, 2048, 1, 4000] + 60 * [2060], 32, 8, 64),
    ([4097, 4096, 4200, 6145] + 60 * [4110], 32, 8, 64),
], ids=lambda x: f"{len(x)}x{max(x)}" if isinstance(x, list) else None)
def test_more_chunks_than_likely(gpu, kind, lens, nq, nkv, d):
    print(f"[case] paged chunks past the likely ones: {kind} {len(lens)}x{max(lens)}", flush=True)
    P = batch(lens, nq, nkv, d, 611)
    B = len(lens)
    K, V = pools(P, nkv, d, kind, 612)
    Q, bt, n = dev(P["q"]), dev(P["bt"].reshape(-1)), dev(P["n"])
    outs = []
    try:
        for forced in (0, 96):
            attn.set_split_chunk(forced)
            O = torch.full((B, nq, d), float("nan"), device="cuda")
            attn.attn_decode_paged(Q, K, V, O, bt, n, None, B, P["max_blocks"], nq, nkv, d, PAGE,
                                   1 / math.sqrt(d), 0)
            outs.append(host(O))
    finally:
        attn.set_split_chunk(0)
    for b in range(B):
        assert normwise_err(outs[0][b], outs[1][b]) < TOL, (b, lens[b])


@pytest.mark.parametrize("kind", ["bf16", "q8"])
@pytest.mark.parametrize("positions", [False, True])
def test_paged_attention_matches_forced_chunks(gpu, kind, positions):
    """Attention only, empty sequences and (positions) query positions behind the
    cache's end under a window: the chunks the device plans and 96-row chunks
    forced from the host agree to the rounding of their sums."""
    print(f"[case] paged chunks against forced ones: {kind} positions={positions}", flush=True)
    lens = [0, 1500, 33, 0, 700, 2048, 1, 129, 64, 3100]
    nq, nkv, d, window = 32, 8, 128, 200 if positions else 0
    P = batch(lens, nq, nkv, d, 411)
    B = len(lens)
    K, V = pools(P, nkv, d, kind, 412)
    pos = dev(np.asarray([max(0, n - 1 - 7 * b) for b, n in enumerate(lens)], np.int32)) \
        if positions else None
    Q, bt, n = dev(P["q"]), dev(P["bt"].reshape(-1)), dev(P["n"])
    s = 1 / math.sqrt(d)
    outs = []
    try:
        for forced in (0, 96):
            attn.set_split_chunk(forced)
            O = torch.full((B, nq, d), float("nan"), device="cuda")
            attn.attn_decode_paged(Q, K, V, O, bt, n, pos, B, P["max_blocks"], nq, nkv, d, PAGE, s,
                                   window)
            outs.append(host(O))
    finally:
        attn.set_split_chunk(0)
    assert np.isfinite(outs[0]).all()
    for b, ln in enumerate(lens):
        if ln == 0:
            assert not outs[0][b].any()
        else:
            assert normwise_err(outs[0][b], outs[1][b]) < TOL, b
