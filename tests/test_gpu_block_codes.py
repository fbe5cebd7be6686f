"""The per-block int8 quantiser's codes over its whole range of scales, bit for
bit the oracle's (IEEE division, half away from zero): ordinary blocks, and
those on either side of the scales it divides element by element for."""

import numpy as np
import pytest
import torch

from oracle import hyq_oracle as O
from tests.gpu_util import to_dev_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factor", [1.0, 3e-3, 2.0 ** -52, 2.0 ** -53, 1e-25, 1e-37, 2.0 ** 62, 2.0 ** 66, 1e30])
def test_block_codes_bit_exact(factor):
    from hyquant_amd.sage_unified import per_block_int8
    rng = np.random.default_rng(8)
    x = rng.standard_normal((1, 2, 4096, 128)).astype(np.float32)
    # half steps of the block's largest value: quotients at and beside the ties
    x[0, 1] = (rng.integers(-254, 255, size=(4096, 128)) * 0.5).astype(np.float32)
    x[0, 1, ::64, 0] = 127.0
    x = O.bf16_round((x * np.float32(factor)).astype(np.float32))
    dev = torch.device("cuda")
    xd = to_dev_bf16(x, dev)
    q8, qs, k8, ks = per_block_int8(xd, xd)
    torch.cuda.synchronize()
    for codes, scales, ref in ((q8, qs, O.per_block_int8(x, np.float32(128 ** -0.5 * O.LOG2E), 128)),
                               (k8, ks, O.per_block_int8(x, 1.0, 64))):
        assert np.array_equal(scales.cpu().numpy().view(np.uint32), ref[1].view(np.uint32))
        assert np.array_equal(codes.cpu().numpy(), ref[0])
