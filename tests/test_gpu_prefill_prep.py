"""The hybrid prefill's preparation launch (lists and K/V statistics together)
at the edges of a statistics chunk, with lists that do and do not repeat an
index, against the float64 oracle at test_gpu_prefill's bound: |out - ref| <=
2e-3 + 2^-10 ref_abs + 2^-8 |ref| (fp16 weights and output rounding)."""

import numpy as np
import pytest
import torch

from oracle import hyq_oracle as O
from tests.gpu_util import to_dev_bf16

pytestmark = pytest.mark.gpu


# 4096 rows fill 32 chunks of 128; one more makes the chunks 256 rows long
@pytest.mark.parametrize("repeats", [False, True], ids=["unique", "repeats"])
@pytest.mark.parametrize("N,W,T", [(127, 64, 9), (128, 1, 127), (129, 96, 33), (4096, 128, 200), (4097, 129, 64)])
def test_prefill_prep_edges(N, W, T, repeats):
    from hyquant_amd.sage_unified import sage_vertical_attention_v2
    print(f"prep N={N} W={W} T={T} repeats={repeats}", flush=True)
    rng = np.random.default_rng(N + T)
    P = N - W
    q, k, v = (O.bf16_round(rng.standard_normal((1, 1, N, 128)).astype(np.float32)) for _ in range(3))
    k = O.bf16_round(k + O.bf16_round(rng.standard_normal((1, 1, 1, 128)).astype(np.float32)))
    v[..., 3] = O.bf16_round(v[..., 3] * 9.0)
    if repeats:
        vidx = rng.integers(-2, P + 2, size=(1, 1, T)).astype(np.int64)
        vidx[..., -1] = vidx[..., 0]
    else:
        vidx = rng.permutation(P)[:T].astype(np.int64).reshape(1, 1, -1)
    dev = torch.device("cuda")
    qd, kd, vd = (to_dev_bf16(x, dev) for x in (q, k, v))
    out = sage_vertical_attention_v2(qd, kd, vd, torch.from_numpy(vidx).to(dev), window_size=W)
    again = sage_vertical_attention_v2(qd, kd, vd, torch.from_numpy(np.sort(vidx, axis=-1)).to(dev), window_size=W)
    torch.cuda.synchronize()
    assert torch.equal(out, again)                    # the order of the indices is of no account
    o = out.float().cpu().numpy()
    ref = O.hybrid_prefill_fp64(q, k, v, vidx, W)
    ref_abs = O.hybrid_prefill_fp64(q, k, v, vidx, W, abs_v=True)
    bad = np.abs(o - ref) > 2e-3 + 2.0 ** -10 * ref_abs + 2.0 ** -8 * np.abs(ref)
    assert not bad.any(), f"{int(bad.sum())} elements, max-abs {float(np.abs(o - ref).max()):.3e}"
