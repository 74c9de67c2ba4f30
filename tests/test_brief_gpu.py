"""Short contexts of one sequence (MI355X only): one chunk up to 64 rows, and
at most 16 chunks a slot merged in the launch up to 2048, at the lines between
them, over every cache type and on 4 to 16 slots; against the oracle.
"""
import numpy as np
import pytest
import torch

import oracle
from conftest import normwise_err
from gpu_util import dev, dev_bf16, host, make_decode
from molot_amd import attn

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("pos", [63, 64, 65, 300, 512, 513, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("nq,nkv,d,kind", [(32, 8, 128, "f32"), (32, 8, 128, "bf16"),
                                           (64, 8, 128, "q8"), (8, 4, 256, "f32"),
                                           (16, 16, 64, "bf16"), (12, 6, 64, "q8"),
                                           (8, 4, 256, "q8")])
def test_brief_decode_step(gpu, nq, nkv, d, kind, pos):
    print(f"[case] brief decode {nq}/{nkv}/{d} {kind} pos={pos}", flush=True)
    p = make_decode(nq, nkv, d, pos, seed=pos + nq, bf16=kind == "bf16")
    if kind == "q8":
        Kq, Vq = (oracle.q8_cache(x, nkv, d) for x in (p.K, p.V))
        K, V = dev(Kq), dev(Vq)
    else:
        K, V = (dev_bf16(p.K), dev_bf16(p.V)) if kind == "bf16" else (dev(p.K), dev(p.V))
    for _ in range(2):  # the second finds the arrival words as the first left them
        q = dev(p.q)
        O = torch.full((nq, d), float("nan"), device="cuda")
        attn.decode_step(q, dev(p.k_new), dev(p.v_new), K, V, O, nq, nkv, d, pos, pos,
                         dev(p.inv_freq), p.scale, 0)
        Kh, Vh = ((host(x.view(torch.int16)).view(np.uint16) if kind == "bf16" else host(x))
                  for x in (K, V))
        row = attn.q8_row_bytes(nkv, d) if kind == "q8" else nkv * d
        R = oracle.attn_decode(host(q), Kh, Vh, nq, nkv, pos + 1, d, p.scale, pos, 0, row, d)
        assert normwise_err(host(O), R) < TOL
