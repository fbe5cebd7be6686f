"""Float64 scores of an fp16 model where a workgroup takes one query head of a
key head, and where it takes all of them: indices equal the oracle's."""

import numpy as np
import pytest
import torch

from oracle import hyq_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,HQ,HK,N,W", [
    (1, 4, 4, 300, 32),        # one query head each
    (1, 6, 2, 1403, 64),       # three, padded to four
    (1, 16, 1, 700, 17),       # sixteen on one key head
    (2, 10, 2, 257, 1),        # five, the last workgroup one row
    (4, 32, 16, 1100, 64),     # 320 workgroups: every CU busy, all heads together
])
def test_selector_fp16_heads_split(B, HQ, HK, N, W):
    from hyquant_amd.vertical import compute_vertical_indices
    print(f"fp16 split B={B} HQ={HQ} HK={HK} N={N} W={W}", flush=True)
    rng = np.random.default_rng(N + HQ)
    rnd = lambda x: x.astype(np.float16).astype(np.float32)
    q, k = (rnd(rng.standard_normal((B, h, N, 128)).astype(np.float32)) for h in (HQ, HK))
    dev = lambda x: torch.from_numpy(x).cuda().half()
    got = compute_vertical_indices(dev(q), dev(k), W, 0.1, kv_repeat=HQ // HK).cpu().numpy()
    assert np.array_equal(got, O.compute_vertical_indices(q, k, W, 0.1, kv_repeat=HQ // HK, fp16=True))
