"""GPU parity of ragged decode on both sides of the lines between the padded
plan and the one formed on the device (bytes, heads, how far the lengths fill
the padded tokens), against the float64 oracle.  The heads share one cache
(head stride 0), so that the padded bytes are not allocated."""

import numpy as np
import pytest
import torch

from oracle import hyq_oracle as O
from tests.gpu_util import to_dev_bf16

pytestmark = pytest.mark.gpu
D = 128


def _inputs(rng, BHK, G, nq, nb, kb, vb):
    """The shared cache on the host and the call's arguments without the lengths."""
    code = lambda bits: rng.integers(-128, 128, (1, nq, D * bits // 8), dtype=np.int8)
    scale = lambda bits: rng.uniform(0.1, 0.4, (1, nq)).astype(np.float16) / np.float16(2 ** (bits - 2))
    rows = lambda: O.bf16_round(rng.standard_normal((1, nb, D)).astype(np.float32))
    host = (code(kb), code(vb), scale(kb), scale(vb), rows(), rows())
    q = O.bf16_round(rng.standard_normal((BHK * G, D)).astype(np.float32))
    up = lambda x: (to_dev_bf16(x, "cuda") if x.dtype == np.float32 else torch.from_numpy(x).cuda()).expand(BHK, *[-1] * (x.ndim - 1))
    return host, q, (to_dev_bf16(q, "cuda"), *(up(x) for x in host))


def _check(out, host, q, lq, lb, G, kb, vb, heads):
    out = out.float().cpu().numpy()
    e = np.zeros((1, 0, D), np.float32)
    for h in heads:
        a, b = int(lq[h]), int(lb[h])
        got = out[h * G:(h + 1) * G]
        if a + b == 0:
            assert not got.any(), h
            continue
        kp, vp, ks, vs, k, v = host
        o = (q[h * G:(h + 1) * G], kp[:, :a], vp[:, :a], ks[:, :a], vs[:, :a], k[:, :b], v[:, :b], e, e, e, e)
        ref = O.decode_fp64(*o, k_bits=kb, v_bits=vb, kv_repeat=G)
        ref_abs = O.decode_fp64(*o, k_bits=kb, v_bits=vb, kv_repeat=G, abs_v=True)
        # 2^-9 sum p|v| / l from P' rounded to bf16, 2^-8 |o| from the output's rounding
        bound = 2e-3 + 2.0 ** -9 * ref_abs + 2.0 ** -8 * np.abs(ref)
        assert np.all(np.abs(got - ref) <= bound), (h, a, b, float((np.abs(got - ref) / bound).max()))


@pytest.mark.parametrize("BHK,G,nq,nb,kb,vb,kind", [
    (64, 4, 11616, 64, 4, 4, "spread"),     # 100.2 MB: planned on the device
    (64, 4, 11584, 64, 4, 4, "spread"),     # 99.96 MB: by the padded lengths
    (64, 4, 28256, 64, 4, 4, "spread"),
    (256, 4, 8000, 333, 4, 4, "spread"),    # the most heads planned on the device
    (257, 4, 8000, 333, 4, 4, "spread"),    # one more
    (64, 16, 40000, 500, 4, 2, "spread"),
    (61, 1, 20000, 31, 8, 8, "spread"),     # heads that are not a multiple of four
    (128, 8, 30000, 0, 2, 2, "spread"),     # no bf16 rows
    (64, 4, 0, 9000, 4, 4, "spread"),       # no prefix
    (64, 4, 30000, 600, 4, 4, 0.59),        # filled to 59%: the device's pieces
    (64, 4, 30000, 600, 4, 4, 0.61),        # to 61%: the padded plan's
    (64, 4, 30000, 600, 4, 4, 1.0),
    (64, 4, 30000, 600, 4, 4, "none"),      # no tokens at all: zeros
    (130, 2, 20000, 64, 4, 4, "one"),       # one long head, the others empty
    (2, 4, 1000000, 1000, 4, 4, "few"),     # more workgroups per head than a plan can have pieces
])
def test_decode_ragged_routes(BHK, G, nq, nb, kb, vb, kind):
    import hyquant_amd as hq
    print(f"ragged BHK={BHK} G={G} nq={nq} nb={nb} K{kb}V{vb} {kind}", flush=True)
    rng = np.random.default_rng(BHK + 7 * G + nq)
    host, q, args = _inputs(rng, BHK, G, nq, nb, kb, vb)
    if kind == "spread":
        lq, lb = (np.floor(n * rng.uniform(0, 1, BHK) ** 4).astype(np.int32) for n in (nq, nb))
        lq[:2], lb[:2] = (0, nq // 2), (0, nb)
    elif isinstance(kind, float):
        lq, lb = (np.full(BHK, int(n * kind), np.int32) for n in (nq, nb))
    elif kind == "few":
        lq, lb = np.array([50001, 17], np.int32), np.array([nb, 0], np.int32)
    else:
        lq, lb = np.zeros(BHK, np.int32), np.zeros(BHK, np.int32)
        if kind == "one":
            lq[BHK // 2], lb[BHK // 2] = nq, nb
    lens = [torch.from_numpy(x).cuda() for x in (lq, lb)]
    out = hq.fused_d_stage_decode_batched(*args, *lens, kb, vb, kv_repeat=G)
    assert torch.equal(out, hq.fused_d_stage_decode_batched(*args, *lens, kb, vb, kv_repeat=G))
    heads = sorted({0, 1, 2, BHK // 2, BHK - 2, BHK - 1} & set(range(BHK)) | set(rng.integers(0, BHK, 10).tolist()))
    _check(out, host, q, lq, lb, G, kb, vb, heads)
    if kind != "one":
        return
    # lengths out of range: past the padded tokens, and negative
    far = [torch.from_numpy(np.where(x > 0, x + 999, x - 5).astype(np.int32)).cuda() for x in (lq, lb)]
    assert torch.equal(out, hq.fused_d_stage_decode_batched(*args, *far, kb, vb, kv_repeat=G))


def test_decode_ragged_replays_on_both_sides_of_the_fill():
    """A captured call follows the lengths of each replay, from nearly empty to
    full and back."""
    import hyquant_amd as hq
    rng = np.random.default_rng(5)
    BHK, G, nq, nb = 64, 4, 30000, 300
    host, q, args = _inputs(rng, BHK, G, nq, nb, 4, 4)
    lq, lb = (torch.zeros(BHK, dtype=torch.int32, device="cuda") for _ in range(2))
    run = lambda: hq.fused_d_stage_decode_batched(*args, lq, lb, 4, 4, kv_repeat=G)
    run()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = run()
    for share in (0.05, 1.0, 0.3, 0.7, 0.0, 0.5):
        a, b = (np.floor(n * share * rng.uniform(0.9, 1.0, BHK)).astype(np.int32) for n in (nq, nb))
        lq.copy_(torch.from_numpy(a))
        lb.copy_(torch.from_numpy(b))
        g.replay()
        got = out.clone()
        assert torch.equal(got, run()), share
        _check(got, host, q, a, b, G, 4, 4, (0, 17, BHK - 1))
