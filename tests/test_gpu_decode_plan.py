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


@pytest.mark.parametrize("BHK,G,nq,nb,kb,vb,kind", [
    (16, 4, 9000, 700, 4, 4, "spread"),    # pieces over lengths of 0 .. 9000
    (9, 16, 6000, 333, 4, 2, "spread"),
    (24, 8, 20000, 1000, 8, 8, "spread"),  # above 48 MB: a quarter more than the resident slots
    (8, 4, 3000, 100, 2, 4, "none"),       # no tokens at all: zeros
    (5, 1, 2000, 0, 4, 4, "spread"),       # no bf16 rows
    (6, 4, 0, 900, 4, 4, "spread"),        # no prefix
    (1024, 2, 70, 9, 4, 4, "spread"),      # the most heads planned on the device
    (1025, 2, 70, 9, 4, 4, "spread"),      # one more: planned by the padded lengths
    (12, 4, 4000, 64, 4, 4, "one"),        # one long head, the others empty
])
def test_decode_ragged_plan(BHK, G, nq, nb, kb, vb, kind):
    import hyquant_amd as hq
    print(f"ragged BHK={BHK} G={G} nq={nq} nb={nb} K{kb}V{vb} {kind}", flush=True)
    rng = np.random.default_rng(BHK + 7 * G + nq)
    D = 128
    st = _state(rng, BHK, nq, nb, 0, 0, kb, vb)
    lq, lb = (rng.integers(0, n + 1, BHK).astype(np.int32) for n in (nq, nb))
    lq[0], lb[0] = nq + 50, nb + 3                      # past the padded length: all of it
    lq[1], lb[1] = (0, 0) if BHK > 5 else (-4, nb)      # an empty head
    if kind == "none":
        lq[:], lb[:] = 0, -1
    elif kind == "one":
        lq[:], lb[:] = 0, 0
        lq[BHK // 2], lb[BHK // 2] = nq, nb
    q = O.bf16_round(rng.standard_normal((BHK * G, D)).astype(np.float32))
    dev = torch.device("cuda")
    t = state_to_device(st, dev)
    args = (to_dev_bf16(q, dev), t["k_packed"], t["v_packed"], t["k_scale"], t["v_scale"], t["k_topk"], t["v_topk"],
            torch.from_numpy(lq).to(dev), torch.from_numpy(lb).to(dev), kb, vb)
    out = hq.fused_d_stage_decode_batched(*args, kv_repeat=G)
    assert torch.equal(out, hq.fused_d_stage_decode_batched(*args, kv_repeat=G))
    out = out.float().cpu().numpy()
    e = np.zeros((1, 0, D), np.float32)
    for h in range(BHK):
        a, b = min(nq, max(0, int(lq[h]))), min(nb, max(0, int(lb[h])))
        got = out[h * G:(h + 1) * G]
        if a + b == 0:
            assert not got.any(), h
            continue
        s = slice(h, h + 1)
        o = (q[h * G:(h + 1) * G], st.k_packed[s, :a], st.v_packed[s, :a], st.k_scale[s, :a], st.v_scale[s, :a],
             st.k_topk[s, :b], st.v_topk[s, :b], e, e, e, e)
        ref = O.decode_fp64(*o, k_bits=kb, v_bits=vb, kv_repeat=G)
        ref_abs = O.decode_fp64(*o, k_bits=kb, v_bits=vb, kv_repeat=G, abs_v=True)
        bound = 2e-3 + 2.0 ** -9 * ref_abs + 2.0 ** -8 * np.abs(ref)
        assert np.all(np.abs(got - ref) <= bound), (h, a, b, float((np.abs(got - ref) / bound).max()))


def test_decode_ragged_plan_replayed():
    """A captured ragged call follows the lengths of each replay."""
    import hyquant_amd as hq
    rng = np.random.default_rng(3)
    BHK, G, nq, nb = 16, 4, 3000, 200
    dev = torch.device("cuda")
    t = state_to_device(_state(rng, BHK, nq, nb, 0, 0, 4, 4), dev)
    q = torch.randn(BHK * G, 128, device=dev).bfloat16()
    lq, lb = (torch.zeros(BHK, dtype=torch.int32, device=dev) for _ in range(2))
    run = lambda: hq.fused_d_stage_decode_batched(q, t["k_packed"], t["v_packed"], t["k_scale"], t["v_scale"],
                                                  t["k_topk"], t["v_topk"], lq, lb, 4, 4, kv_repeat=G)
    run()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = run()
    for i in range(4):
        lq.copy_(torch.from_numpy(rng.integers(0, nq + 1, BHK).astype(np.int32)))
        lb.copy_(torch.from_numpy(rng.integers(0, nb + 1, BHK).astype(np.int32)))
        g.replay()
        got = out.clone()
        assert torch.equal(got, run()), i


def test_decode_ragged_workspace_of_the_padded_plan():
    """A workspace sized without the lengths is still enough to run with them."""
    import ctypes
    from hyquant_amd import _lib
    from hyquant_amd.decode_d_stage import decode_params
    rng = np.random.default_rng(4)
    BHK, G, nq, nb = 4, 4, 500, 40
    dev = torch.device("cuda")
    t = state_to_device(_state(rng, BHK, nq, nb, 0, 0, 4, 4), dev)
    q = torch.randn(BHK * G, 128, device=dev).bfloat16()
    lq = torch.tensor([500, 0, 33, 264], dtype=torch.int32, device=dev)
    lb = torch.tensor([7, 40, 0, 21], dtype=torch.int32, device=dev)
    e = t["k_topk"][:, :0]
    args = (q, t["k_packed"], t["v_packed"], t["k_scale"], t["v_scale"], t["k_topk"], t["v_topk"], e, e, e, e, 4, 4, G)
    L = _lib.lib()
    outs, sizes = [], []
    for sized_with in (dict(), dict(lens_q=lq, lens_s0=lb)):
        p, keep, _ = decode_params(*args, **sized_with)
        n = L.hyq_decode_workspace_size(ctypes.byref(p))
        p, keep, out = decode_params(*args, lens_q=lq, lens_s0=lb)
        ws = torch.zeros(n, dtype=torch.uint8, device=dev)
        _lib.check(L.hyq_decode_hybrid(ctypes.byref(p), ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream),
                   "hyq_decode_hybrid")
        torch.cuda.synchronize()
        outs.append(out.float())
        sizes.append(n)
    assert sizes[0] < sizes[1]
    # the two plans differ in the order of the sums only: two roundings to bf16
    assert torch.all((outs[0] - outs[1]).abs() <= 2.0 ** -7 * outs[0].abs() + 1e-3)
