"""CPU checks of the staging buffers: an append whose keys and values autograd
records is an ordinary copy, under whatever grad mode the freeze ran."""

import pytest
import torch

from hyquant_amd import d_stage_kv_cache as kc


def _frozen(BH, D):
    layer = kc.DStageLayerCache(0)
    layer.phase = "decode"
    layer._B, layer._H_KV, layer._D = 1, BH, D
    layer._staging_buf_k, layer._staging_buf_v = kc._staging_buffers(BH, D, torch.device("cpu"), torch.bfloat16)
    return layer


@pytest.mark.parametrize("frozen_in", [torch.enable_grad, torch.no_grad])
def test_append_of_keys_that_require_grad(frozen_in):
    BH, D = 3, 16
    with frozen_in():
        layer = _frozen(BH, D)
    g = torch.Generator().manual_seed(0)
    rows = [torch.randn(1, BH, 1, D, generator=g).bfloat16() for _ in range(4)]
    with torch.enable_grad():
        for k, v in (rows[:2], rows[2:]):
            layer.append_staging(k.clone().requires_grad_(), v.clone().requires_grad_())
    assert layer._staging_ptr == 2 and layer.get_seq_length() == 2
    for buf, (a, b) in ((layer._staging_buf_k, rows[0::2]), (layer._staging_buf_v, rows[1::2])):
        assert torch.equal(buf.detach()[:, :2], torch.cat([a[0], b[0]], 1))
        assert not buf.detach()[:, 2:].any()


def test_staging_buffers_are_tensors_of_their_own():
    k, v = kc._staging_buffers(2, 16, torch.device("cpu"), torch.float16)
    assert not k._is_view() and not v._is_view()
    assert k.shape == v.shape == (2, 128, 16) and k.is_contiguous() and v.is_contiguous()
    before = v._version
    k.fill_(1.0)
    assert v._version == before and not v.any()
