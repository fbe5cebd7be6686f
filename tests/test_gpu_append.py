"""The staging append (hyq_append_rows) and the layer cache's native decode
step against tensor copies and the checked call."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,n,D,dtype,order", [
    (1, 8, 1, 128, torch.bfloat16, "token"), (3, 2, 5, 128, torch.float16, "head"), (1, 1, 128, 64, torch.bfloat16, "head"),
    (2, 3, 7, 256, torch.float16, "token"),
])
def test_append_rows_equals_copies(B, H, n, D, dtype, order):
    import hyquant_amd.decode_d_stage as dd
    fx = dd._load_fast_ext()
    assert fx, "the eager-call extension is not built"
    shape = (B, n, H, D) if order == "token" else (B, H, n, D)
    k, v = (torch.randn(shape, device="cuda").to(dtype) for _ in range(2))
    if order == "token":
        k, v = k.transpose(1, 2), v.transpose(1, 2)
    bk, bv = (torch.full((B * H, 128, D), 7.0, dtype=dtype, device="cuda") for _ in range(2))
    ek, ev = bk.clone(), bv.clone()
    row = 128 - n
    stream = torch.cuda.current_stream().cuda_stream
    assert fx.append(k, v, bk, bv, row, stream) == 0
    ek[:, row:].copy_(k.reshape(B * H, n, D))
    ev[:, row:].copy_(v.reshape(B * H, n, D))
    assert torch.equal(bk, ek) and torch.equal(bv, ev)
    # declined, nothing written: past the end, another type, channels apart, recorded by autograd
    assert fx.append(k, v, bk, bv, row + 1, stream) == -1
    assert fx.append(k.float(), v.float(), bk, bv, 0, stream) == -1
    assert fx.append(torch.randn(B, H, n, 2 * D, device="cuda").to(dtype)[..., ::2], v, bk, bv, 0, stream) == -1
    assert fx.append(k.clone().requires_grad_(), v, bk, bv, 0, stream) == -1
    assert torch.equal(bk, ek) and torch.equal(bv, ev)


@pytest.mark.parametrize("B,HQ,HK,dtype", [(1, 8, 2, torch.bfloat16), (2, 8, 8, torch.float16)])
def test_layer_steps_equal_the_checked_path(B, HQ, HK, dtype, monkeypatch):
    """130 steps across a flush, once with the extension and once without:
    equal outputs and equal caches, bit for bit."""
    import hyquant_amd.decode_d_stage as dd
    from hyquant_amd.d_stage_kv_cache import DStageLayerCache
    assert dd._load_fast_ext()
    N, W, D, steps = 300, 64, 128, 130
    torch.manual_seed(B)
    rnd = lambda h, n: torch.randn(B, n, h, D, device="cuda").to(dtype).transpose(1, 2)
    q, k, v = rnd(HQ, N), rnd(HK, N), rnd(HK, N)
    new = [(rnd(HQ, 1), rnd(HK, 1), rnd(HK, 1)) for _ in range(steps)]
    got = []
    for fast in (True, False):
        if not fast:
            monkeypatch.setattr(dd, "_FX", False)
        c = DStageLayerCache(0, 4, 4, window_size=W)
        c.update_prefill(k, v)
        c.save_query_tail(q)
        c.freeze(kv_repeat=HQ // HK)
        outs = []
        for a, b, d in new:
            c.append_staging(b, d)
            outs.append(c.decode_attention(a, HQ // HK))
        got.append([torch.cat(outs, 2), c.k_quant_packed, c.v_scale, c._staging_buf_k[:, :c._staging_ptr].clone()])
        assert c.get_seq_length() == N + steps and c._staging_ptr == steps - 128
    for x, y in zip(*got):
        assert x.shape == y.shape and torch.equal(x, y)


def _frozen(B, HQ, HK, dtype, N=300, W=64, D=128):
    from hyquant_amd.d_stage_kv_cache import DStageLayerCache
    torch.manual_seed(B + HQ)
    rnd = lambda h, n: torch.randn(B, n, h, D, device="cuda").to(dtype).transpose(1, 2)
    c = DStageLayerCache(0, 4, 4, window_size=W)
    c.update_prefill(rnd(HK, N), rnd(HK, N))
    c.save_query_tail(rnd(HQ, N))
    c.freeze(kv_repeat=HQ // HK)
    for _ in range(3):
        c.append_staging(rnd(HK, 1), rnd(HK, 1))
    return c, rnd(HQ, 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_native_step_takes_a_layer_and_declines_the_rest(dtype):
    import hyquant_amd.decode_d_stage as dd
    B, HQ, HK, D = 2, 8, 2, 128
    c, q = _frozen(B, HQ, HK, dtype)
    ref = c.decode_attention(q, HQ // HK)              # (and the stream's workspace is there)
    stream = torch.cuda.current_stream().cuda_stream
    ws = dd._ws_raw[(q.get_device(), stream)]

    def step(q=q, batch=B, nq=c._kstore.n, ns=c._staging_ptr, repeat=HQ // HK):
        return dd._FX.decode_cache(q, batch, c._kstore.packed, c._vstore.packed, c._kstore.scale, c._vstore.scale, nq,
                                   c.k_topk, c.v_topk, c._staging_buf_k, c._staging_buf_v, ns, c.k_window, c.v_window, 4,
                                   4, repeat, stream, *ws)

    st, out = step()
    assert st == 0 and out.shape == (B, HQ, 1, D) and torch.equal(out, ref)
    wide = torch.zeros(B, HQ + 1, 1, D, device="cuda", dtype=dtype)[:, :HQ].copy_(q)
    for bad in (dict(q=wide), dict(q=q.reshape(1, B * HQ, 1, D)), dict(q=q[:, :, 0]), dict(repeat=HQ // HK + 1), dict(batch=1),
                dict(nq=c._kstore.packed.shape[1] + 1), dict(ns=c._staging_buf_k.shape[1] + 1), dict(nq=-1), dict(ns=-1)):
        assert step(**bad)[0] == -1, list(bad)
    # what the native step declines has the same result, in the cache's shape
    assert torch.equal(c.decode_attention(wide, HQ // HK), ref)
    assert torch.equal(c.decode_attention(q.reshape(1, B * HQ, 1, D), HQ // HK), ref)


def test_append_staging_copies_rows_that_are_not_16_byte_aligned():
    import hyquant_amd.decode_d_stage as dd
    B, HK, D = 2, 2, 128
    c, _ = _frozen(B, 8, HK, torch.bfloat16)
    rows = [torch.randn(B * HK * D + 1, device="cuda").bfloat16()[1:].view(B, HK, 1, D) for _ in range(2)]
    at = c._staging_ptr
    assert dd._FX.append(*rows, c._staging_buf_k, c._staging_buf_v, at, torch.cuda.current_stream().cuda_stream) not in (0, -1)
    c.append_staging(*rows)
    assert c._staging_ptr == at + 1
    assert torch.equal(c._staging_buf_k[:, at], rows[0].view(B * HK, D))
    assert torch.equal(c._staging_buf_v[:, at], rows[1].view(B * HK, D))


def test_append_staging_takes_recorded_rows():
    """Keys that require grad, under grad mode: declined, then copied."""
    B, HK, D = 2, 2, 128
    c, _ = _frozen(B, 8, HK, torch.bfloat16)
    rows = [torch.randn(B, HK, 1, D, device="cuda").bfloat16().requires_grad_() for _ in range(2)]
    at = c._staging_ptr
    with torch.enable_grad():
        c.append_staging(*rows)
    assert c._staging_ptr == at + 1
    assert torch.equal(c._staging_buf_k[:, at].detach(), rows[0].detach().view(B * HK, D))
