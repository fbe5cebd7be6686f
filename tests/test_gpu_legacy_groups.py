"""GPU parity of the legacy-format decode through the C ABI where its walk of
the scale groups can go wrong: groups that are not a multiple of 32 tokens,
groups longer than the prefix, prefixes that end inside a chunk or a block,
both block sizes, and K scales spread over 2^17 between channels."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import hyq_oracle as O
from tests.gpu_util import to_dev_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BHK,R,N,group,kb,vb,spread", [
    (3, 4, 1000, 16, 4, 4, False),       # half-filled chunks
    (2, 16, 33, 128, 2, 2, False),       # one token past a chunk
    (3, 1, 1, 128, 4, 2, False),
    (3, 4, 129, 4096, 4, 4, True),       # the group longer than the prefix
    (3, 4, 700, 96, 4, 2, False),        # three chunks a group
    (2, 4, 1200, 1184, 2, 4, False),     # 37 chunks in the first, one in the second
    (128, 2, 1100, 112, 4, 4, False),    # blocks of four chunks, the last 16 tokens
    (130, 4, 1151, 128, 2, 4, True),     # blocks of four, one token short of a chunk
    (128, 8, 1153, 256, 4, 2, False),    # two blocks per group, one token in the last
])
def test_legacy_group_walk(BHK, R, N, group, kb, vb, spread):
    from hyquant_amd import _lib
    print(f"legacy groups BHK={BHK} R={R} N={N} group={group} K{kb}V{vb}", flush=True)
    L = _lib.lib()
    rng = np.random.default_rng(BHK + N + group)
    D, T = 128, 5
    G = -(-N // group)
    kp = rng.integers(0, 256, (BHK, N, 16 * kb), dtype=np.uint8)
    vp = rng.integers(0, 256, (BHK, N, 16 * vb), dtype=np.uint8)
    mag = 2.0 ** rng.uniform(-20, -3, (BHK, G, D)) if spread else rng.uniform(0.01, 0.12, (BHK, G, D))
    ks = (mag * rng.choice([-1.0, 1.0], (BHK, G, D))).astype(np.float16)
    vs = rng.uniform(-0.12, 0.12, (BHK, G, D)).astype(np.float16)
    f = lambda n: O.bf16_round(rng.standard_normal((BHK, n, D)).astype(np.float32))
    kt, vt = f(T), f(T)
    e = np.zeros((BHK, 0, D), np.float32)
    q = O.bf16_round(rng.standard_normal((BHK * R, D)).astype(np.float32))
    u = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    keep = [u(kp), u(vp), u(ks), u(vs), to_dev_bf16(kt, "cuda"), to_dev_bf16(vt, "cuda"), to_dev_bf16(q, "cuda")]
    out = torch.empty(BHK * R, D, dtype=torch.bfloat16, device="cuda")
    p = _lib.LegacyParams()
    p.q, p.q_stride, p.out, p.out_stride = keep[6].data_ptr(), D, out.data_ptr(), D
    p.k_codes, p.kc_stride_bh, p.kc_stride_n = keep[0].data_ptr(), N * 16 * kb, 16 * kb
    p.v_codes, p.vc_stride_bh, p.vc_stride_n = keep[1].data_ptr(), N * 16 * vb, 16 * vb
    p.k_scale, p.ks_stride_bh, p.ks_stride_g = keep[2].data_ptr(), G * D, D
    p.v_scale, p.vs_stride_bh, p.vs_stride_g = keep[3].data_ptr(), G * D, D
    p.n, p.group, p.k_bits, p.v_bits = N, group, kb, vb
    p.seg_k[0], p.seg_v[0], p.seg_k_stride_bh[0], p.seg_v_stride_bh[0], p.seg_n[0] = (
        keep[4].data_ptr(), keep[5].data_ptr(), T * D, T * D, T)
    p.bh_kv, p.kv_repeat, p.head_dim, p.sm_scale = BHK, R, D, D ** -0.5
    need = L.hyq_decode_legacy_workspace_size(ctypes.byref(p))
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    st = L.hyq_decode_legacy(ctypes.byref(p), ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    assert st == 0, L.hyq_last_error()
    got = out.float().cpu().numpy()
    args = (q, kp, vp, ks, vs, kt, vt, e, e, e, e)
    ref = O.legacy_decode_fp64(*args, k_bits=kb, v_bits=vb, kv_repeat=R, group=group)
    ref_abs = O.legacy_decode_fp64(*args, k_bits=kb, v_bits=vb, kv_repeat=R, group=group, abs_v=True)
    # P and the output rounded to bf16, the folded query to fp16 (2^-12 of a
    # score of magnitude below 4 moves a weight by less than 2^-9)
    bound = 2e-3 + 2.0 ** -8 * ref_abs + 2.0 ** -8 * np.abs(ref)
    assert np.all(np.abs(got - ref) <= bound), float((np.abs(got - ref) / bound).max())
