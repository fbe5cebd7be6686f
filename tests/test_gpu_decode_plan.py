"""GPU parity of the decode kernel at the piece counts each rule of its plan
picks (hyquant_amd/csrc/decode.hip, make_plan): the edges of the rules in KV
heads, bytes and heads per group, against the float64 oracle."""

import numpy as np
import pytest
import torch

from oracle import hyq_oracle as O
from tests.gpu_util import state_to_device, to_dev_bf16

pytestmark = pytest.mark.gpu


def _state(rng, BHK, nq, T, S, W, kb, vb):
    D = 128
    b = lambda n: O.bf16_round(rng.standard_normal((BHK, n, D)).astype(np.float32))
    code = lambda bits: rng.integers(-128, 128, (BHK, nq, D * bits // 8), dtype=np.int8)
    scale = lambda bits: rng.uniform(0.1, 0.4, (BHK, nq)).astype(np.float16) / np.float16(2 ** (bits - 2))
    st = O.DecodeState(code(kb), code(vb), scale(kb), scale(vb), b(T), b(T), b(W), b(W),
                       np.zeros((BHK, 128, D), np.float32), np.zeros((BHK, 128, D), np.float32), k_bits=kb, v_bits=vb)
    st.k_ring[:, :S] = b(S)
    st.v_ring[:, :S] = b(S)
    st.ring_ptr = S
    return st


@pytest.mark.parametrize("BHK,G,nq,T,S,W,kb,vb", [
    (2, 16, 900, 40, 7, 128, 4, 4),        # few heads, modelled piece count
    (31, 8, 700, 33, 127, 128, 4, 2),      # the last batch below 32 heads
    (32, 4, 31, 1, 1, 1, 4, 4),            # 32 heads, segments of one unit each
    (64, 4, 1500, 61, 64, 128, 8, 8),      # the most heads of the modelled range
    (65, 4, 500, 25, 64, 128, 4, 4),       # above it
    (20, 16, 21500, 900, 64, 256, 4, 4),   # 60 MB and 20 heads at G = 16: twelve pieces
    (19, 16, 21500, 900, 64, 256, 2, 4),   # one head fewer
])
def test_decode_plan_edges(BHK, G, nq, T, S, W, kb, vb):
    import hyquant_amd as hq
    print(f"plan BHK={BHK} G={G} nq={nq} T={T} S={S} W={W} K{kb}V{vb}", flush=True)
    rng = np.random.default_rng(BHK * 1000 + G + nq)
    st = _state(rng, BHK, nq, T, S, W, kb, vb)
    q = O.bf16_round(rng.standard_normal((BHK * G, 128)).astype(np.float32))
    dev = torch.device("cuda")
    t = state_to_device(st, dev)
    out = hq.fused_d_stage_decode(to_dev_bf16(q, dev), t["k_packed"], t["v_packed"], t["k_scale"], t["v_scale"],
                                  t["k_topk"], t["v_topk"], t["k_staging"], t["v_staging"], t["k_window"],
                                  t["v_window"], kb, vb, kv_repeat=G).float().cpu().numpy()
    ref = O.decode_fp64_state(q, st, G)
    ref_abs = O.decode_fp64_state(q, st, G, abs_v=True)
    # 2^-9 sum p|v| / l from P' rounded to bf16, 2^-8 |o| from the output's rounding
    bound = 2e-3 + 2.0 ** -9 * ref_abs + 2.0 ** -8 * np.abs(ref)
    assert np.all(np.abs(out - ref) <= bound), float((np.abs(out - ref) / bound).max())
