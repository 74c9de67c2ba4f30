"""The 32-row prefill kernels lose no accuracy against the kernels they stand in
for (MI355X only): their error against a float64 attention over the same cache is
no larger than that of the path a smaller prompt takes (the presplit switch off).
"""
import math

import numpy as np
import pytest
import torch

from gpu_util import dev, host
from molot_amd import attn
from molot_amd.synth import Stream, bf16_to_f32
from test_d512_gpu import caches, on_dev

pytestmark = pytest.mark.gpu

# (nq, nkv, d, M, n0, kind)
SHAPES = [
    (8, 2, 512, 300, 9000, "f32"),
    (8, 2, 512, 300, 9000, "q8"),
    (8, 2, 512, 700, 0, "bf16"),
    (32, 8, 128, 300, 900, "f32"),
    (32, 8, 128, 300, 900, "bf16"),
    (32, 8, 128, 1024, 0, "f32"),
    (32, 8, 64, 300, 8000, "f32"),
]


def values64(X, nkv, d):
    """A token-major cache's values, exactly."""
    if X.dtype == np.uint8:
        codes = X[:, :nkv * d].copy().view(np.int8).reshape(-1, nkv, d)
        scales = X[:, nkv * d:nkv * d + 4 * nkv].copy().view(np.float32).reshape(-1, nkv, 1)
        return (codes.astype(np.float64) * scales).reshape(X.shape[0], nkv * d)
    return (bf16_to_f32(X) if X.dtype == np.uint16 else X).astype(np.float64)


def attend64(Q, K, V, nq, nkv, d, n0):
    """Causal attention in 64 bits, on the GPU."""
    Q, K, V = (torch.from_numpy(np.ascontiguousarray(x, np.float64)).cuda() for x in (Q, K, V))
    M, N = Q.shape[0], K.shape[0]
    K, V = K.view(N, nkv, d), V.view(N, nkv, d)
    dead = torch.arange(N, device="cuda")[None] > n0 + torch.arange(M, device="cuda")[:, None]
    O = torch.empty_like(Q)
    for h in range(nq):
        kv = h // (nq // nkv)
        s = (Q[:, h].contiguous() @ K[:, kv].T.contiguous()) / math.sqrt(d)
        O[:, h] = s.masked_fill_(dead, -math.inf).softmax(-1) @ V[:, kv].contiguous()
    return O.cpu().numpy()


@pytest.mark.parametrize("shape", SHAPES,
                         ids=[f"{s[0]}q{s[1]}kv_d{s[2]}_M{s[3]}_n{s[4]}_{s[5]}" for s in SHAPES])
def test_error_no_larger_than_the_smaller_prompts_path(gpu, shape):
    nq, nkv, d, M, n0, kind = shape
    print(f"[case] prefill accuracy {shape}", flush=True)
    st = Stream(801 + d + n0)
    Q = st.normal((M, nq, d))
    K, V = caches(st, n0 + M, nkv, d, kind)
    R = attend64(Q, values64(K, nkv, d), values64(V, nkv, d), nq, nkv, d, n0)
    Qd, Kd, Vd = dev(Q), on_dev(K), on_dev(V)
    err = []
    try:
        for on in (True, False):
            attn.set_prefill_presplit(on)
            O = torch.empty((M, nq, d), device="cuda")
            attn.attn_prefill_gqa(Qd, Kd, Vd, O, nq, nkv, M, n0 + M, d, 1 / math.sqrt(d), n0, 0)
            err.append(float(np.linalg.norm(host(O) - R) / np.linalg.norm(R)))
    finally:
        attn.set_prefill_presplit(True)
    print(f"error against 64 bits {err[0]:.3e}, the smaller prompts' path {err[1]:.3e}", flush=True)
    assert err[0] <= err[1]
