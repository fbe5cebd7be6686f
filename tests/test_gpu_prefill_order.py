"""The order in which the hybrid prefill takes its query blocks: every head of
a call has to come out bit for bit as in a call of its own (a head's result
does not depend on the others), whatever share of the heads fills whole XCDs."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,N", [
    (1, 100),        # one block: seven XCDs idle
    (3, 700),        # fewer heads than XCDs: blocks dealt to all
    (8, 129),        # one head per XCD
    (9, 1300),       # one head beyond
    (40, 600),       # five per XCD, one group
    (31, 257),       # three per XCD and seven dealt
    (24, 12800),     # 100 blocks: groups of two heads and one
    (16, 33000),     # 258 blocks: one head at a time
])
@pytest.mark.parametrize("pv_mode", ["fp16", "fp8"])
def test_prefill_heads_equal_single_calls(heads, N, pv_mode):
    from hyquant_amd.sage_unified import sage_vertical_attention_v2
    print(f"order heads={heads} N={N} {pv_mode}", flush=True)
    W, dev = 64, torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(heads + N)
    q, k, v = (torch.randn(1, heads, N, 128, device=dev, generator=g, dtype=torch.bfloat16) for _ in range(3))
    T = (N - W) // 20
    vidx = torch.stack([torch.randperm(N - W, device=dev, generator=g)[:T] for _ in range(heads)])[None]
    run = lambda s: sage_vertical_attention_v2(q[:, s], k[:, s], v[:, s], vidx[:, s], window_size=W, pv_mode=pv_mode)
    out = run(slice(None))
    for h in sorted({0, 1, heads // 2, 7, 8, heads - 2, heads - 1} & set(range(heads))):
        assert torch.equal(out[:, h:h + 1], run(slice(h, h + 1))), h
