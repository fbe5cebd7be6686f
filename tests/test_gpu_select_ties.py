"""The selector where many keys score alike: buckets of the counting rank on
both sides of its bitmap limit, several of them in one row, cut by the top-k,
and fewer key rows per workgroup than a full one."""

import numpy as np
import pytest
import torch

from oracle import hyq_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,groups,rho,fp16", [
    (3000, [128], 0.05, False), (3000, [129], 0.05, False), (3000, [140, 200, 131], 0.12, False),
    (9000, [700, 700], 0.1, True), (33000, [1500, 300], 0.05, False), (300, [270], 0.5, True),
])
def test_selector_equal_scores(N, groups, rho, fp16):
    from hyquant_amd.vertical import compute_vertical_indices
    print(f"select ties N={N} groups={groups} rho={rho} fp16={fp16}", flush=True)
    B, HQ, HK, W, D = 1, 4, 2, 16, 128
    rng = np.random.default_rng(N + len(groups))
    rnd = (lambda x: x.astype(np.float16).astype(np.float32)) if fp16 else O.bf16_round
    q = rnd(rng.standard_normal((B, HQ, W, D)).astype(np.float32))
    k = rnd((0.2 * rng.standard_normal((B, HK, N, D))).astype(np.float32))
    u = q.mean(axis=(1, 2))
    pos = rng.permutation(N - W)
    at = 0
    for i, n in enumerate(groups):                      # n copies of one key along the mean query
        k[:, :, pos[at:at + n]] = rnd(((2.0 + i) * u).astype(np.float32))[:, None, None, :]
        at += n
    dt = torch.float16 if fp16 else torch.bfloat16
    dev = lambda x: torch.from_numpy(x).cuda().to(dt)
    got = compute_vertical_indices(dev(q), dev(k), W, rho, kv_repeat=HQ // HK).cpu().numpy()
    exp = O.compute_vertical_indices(q, k, W, rho, kv_repeat=HQ // HK, fp16=fp16)
    assert np.array_equal(got, exp)
