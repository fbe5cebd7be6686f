"""The hybrid prefill where a query block's runs of tiles begin and end: rest
tiles, then vertical and window tiles in one run.  Against the float64 oracle
at test_gpu_prefill's bound: |out - ref| <= 2e-3 + 2^-10 ref_abs + 2^-8 |ref|
(fp16 weights and output rounding)."""

import numpy as np
import pytest
import torch

from oracle import hyq_oracle as O
from tests.gpu_util import to_dev_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,W,T", [
    (64, 64, 0),       # one window tile
    (129, 1, 64),      # no whole window tile; vertical entries up to one tile
    (300, 64, 63),     # the vertical tile one short of full
    (300, 64, 64),     # full
    (300, 64, 65),     # one more
    (192, 64, 128),    # every prefix position vertical: no rest tiles
    (513, 128, 320),   # five vertical tiles before the last block's window
    (640, 512, 2),     # window tiles in the majority
])
@pytest.mark.parametrize("entry", ["int8", "fp8qk"])
def test_prefill_run_boundaries(N, W, T, entry):
    from hyquant_amd import sage_unified as su
    print(f"runs {entry} N={N} W={W} T={T}", flush=True)
    rng = np.random.default_rng(N + 7 * T)
    q, k, v = (O.bf16_round(rng.standard_normal((1, 2, N, 128)).astype(np.float32)) for _ in range(3))
    # rising keys: the running maximum moves again and again, across the runs too
    k = O.bf16_round(k * np.linspace(0.5, 3.0, N, dtype=np.float32)[:, None])
    vidx = np.stack([rng.permutation(N - W)[:T] for _ in range(2)]).astype(np.int64).reshape(1, 2, T)
    dev = torch.device("cuda")
    fn = su.sage_vertical_attention_v2 if entry == "int8" else su.sage_vertical_attention_v2_fp8
    out = fn(*(to_dev_bf16(x, dev) for x in (q, k, v)), torch.from_numpy(vidx).to(dev), window_size=W)
    o = out.float().cpu().numpy()
    mode = dict(qk_mode="int8" if entry == "int8" else "fp8")
    ref = O.hybrid_prefill_fp64(q, k, v, vidx, W, **mode)
    ref_abs = O.hybrid_prefill_fp64(q, k, v, vidx, W, abs_v=True, **mode)
    bad = np.abs(o - ref) > 2e-3 + 2.0 ** -10 * ref_abs + 2.0 ** -8 * np.abs(ref)
    assert not bad.any(), f"{int(bad.sum())} elements, max-abs {float(np.abs(o - ref).max()):.3e}"
