"""CPU checks of the decode plans' pieces, read back from the workspace sizes
(arrival counters, then an (m, l) pair and 128 sums per query head and piece)."""

import pytest

COUNTERS = 16384 * 128


def _pieces(size, bh, G):
    """Pieces per head of a workspace of `size` bytes."""
    r = lambda x: (x + 255) // 256 * 256
    fit = [k for k in range(1, 257) if COUNTERS + r(8 * bh * k * G) + r(512 * bh * k * G) == size]
    assert len(fit) == 1, (size, fit)
    return fit[0]


@pytest.mark.parametrize("G", [1, 4, 8, 16])
@pytest.mark.parametrize("bh", [1, 20, 64, 65, 128, 2048, 16384])
@pytest.mark.parametrize("stride,group", [(4096, 128), (4096, 16), (4096, 1 << 24), (2048, 112), (512, 128), (64, 128)])
def test_legacy_pieces_stay_within_32_bit_offsets(bh, G, stride, group):
    """A piece's rows (and 640 rows of look-ahead) have to span less than 2^32
    bytes: its descriptors and offsets are 32 bits wide.  A prefix of n tokens
    in k pieces has one of at least n / k."""
    from hyquant_amd import _lib
    L = _lib.lib()
    p = _lib.LegacyParams()
    p.q, p.q_stride, p.out, p.out_stride = 256, 128, 512, 128
    p.k_codes, p.v_codes, p.k_scale, p.v_scale = 4096, 8192, 16384, 32768
    p.kc_stride_n, p.vc_stride_n = stride, 64
    p.ks_stride_g = p.vs_stride_g = 128
    p.group, p.k_bits, p.v_bits = group, 4, 4
    p.bh_kv, p.kv_repeat, p.head_dim, p.sm_scale = bh, G, 128, 128 ** -0.5
    for n in (1000, 1 << 20, (1 << 21) + 17, 1 << 24):
        p.n = n
        for swap in (False, True):
            if swap:
                p.kc_stride_n, p.vc_stride_n = 64, stride
            k = _pieces(L.hyq_decode_legacy_workspace_size(p), bh, G)
            # pieces are whole blocks of at most 128 tokens, so the largest is
            # at most a block above the mean
            assert (n / k + 128 + 640) * stride <= 2 ** 32, (n, k)


@pytest.mark.parametrize("bh,G", [(8, 4), (64, 16), (2048, 4), (16384, 16)])
def test_legacy_segments_stay_within_32_bit_offsets(bh, G):
    """2^24 rows of 256 bytes fill 32 bits: such a segment has two pieces at least."""
    from hyquant_amd import _lib
    L = _lib.lib()
    p = _lib.LegacyParams()
    p.q, p.q_stride, p.out, p.out_stride = 256, 128, 512, 128
    p.k_bits = p.v_bits = 4
    p.seg_k[0], p.seg_v[0], p.seg_n[0] = 65536, 131072, 1 << 24
    p.bh_kv, p.kv_repeat, p.head_dim, p.sm_scale = bh, G, 128, 128 ** -0.5
    assert _pieces(L.hyq_decode_legacy_workspace_size(p), bh, G) >= 2


@pytest.mark.parametrize("bh,G,n,kb,vb,good", [
    # kernel time by pieces per head, us
    (40, 4, 5151, 4, 2, (9, 10)),            # 6: 13.5, 9: 12.1, 10: 11.5, 11: 13.5
    (48, 8, 10000, 4, 2, (7, 8, 9)),         # 10: 23.4, 7: 20.6, 9: 19.8
    (32, 8, 13001, 4, 2, (10, 11, 12, 13)),  # 7: 21.4, 10: 19.1, 13: 18.3
    (48, 4, 3600, 4, 4, (7, 8)),             # 6: 12.8, 7: 11.4, 8: 11.1, 9: 12.2
    (32, 16, 30000, 8, 8, (9, 10)),          # 8: 61.6, 9: 57.7, 10: 54.3, 12: 73.2
    (64, 16, 3600, 8, 8, (7,)),              # 6: 22.9, 7: 20.4, 8: 24.2, 12: 24.7
    (48, 16, 16384, 4, 4, (7, 12)),          # 7: 30.2, 12: 29.9, 1.25 rounds: 33.5
    (8, 4, 8192, 4, 4, (26,)),               # equal bytes, 0.8 pieces per CU
])
def test_decode_piece_counts_are_the_fast_ones(bh, G, n, kb, vb, good):
    """On a device of 256 CUs (also what is assumed where there is none)."""
    from hyquant_amd import _lib
    L = _lib.lib()
    p = _lib.DecodeParams()
    p.q, p.q_stride, p.out, p.out_stride = 256, 128, 512, 128
    p.k_packed, p.v_packed, p.k_scale, p.v_scale = 4096, 8192, 16384, 32768
    p.kp_stride_n, p.vp_stride_n, p.n_quant = 16 * kb, 16 * vb, n
    for s, m in enumerate((n // 20, 64, 128)):
        p.seg_k[s], p.seg_v[s], p.seg_n[s] = 65536, 131072, m
        p.seg_k_stride_n[s] = p.seg_v_stride_n[s] = 128
    p.bh_kv, p.kv_repeat, p.head_dim, p.k_bits, p.v_bits, p.sm_scale = bh, G, 128, kb, vb, 128 ** -0.5
    assert _pieces(L.hyq_decode_workspace_size(p), bh, G) in good


@pytest.mark.parametrize("bh,G,n,bits,good", [
    (24, 4, 5151, 2, (16, 17)),              # 9: 16.8, 12: 13.4, 16: 11.8, 17: 11.9
    (32, 4, 3600, 2, (12, 13, 14, 15)),      # 8: 15.6, 12: 12.0, 14: 9.6
    (8, 4, 2500, 4, (28, 30, 32)),           # 14: 8.8, 20: 8.0, 30: 7.2, 32: 7.1, 48: 8.7
])
def test_legacy_piece_counts_are_the_fast_ones(bh, G, n, bits, good):
    from hyquant_amd import _lib
    L = _lib.lib()
    p = _lib.LegacyParams()
    p.q, p.q_stride, p.out, p.out_stride = 256, 128, 512, 128
    p.k_codes, p.v_codes, p.k_scale, p.v_scale = 4096, 8192, 16384, 32768
    p.kc_stride_n = p.vc_stride_n = 16 * bits
    p.ks_stride_g = p.vs_stride_g = 128
    p.n, p.group, p.k_bits, p.v_bits = n, 128, bits, bits
    for s, m in enumerate((n // 20, 64, 128)):
        p.seg_k[s], p.seg_v[s], p.seg_n[s] = 65536, 131072, m
    p.bh_kv, p.kv_repeat, p.head_dim, p.sm_scale = bh, G, 128, 128 ** -0.5
    assert _pieces(L.hyq_decode_legacy_workspace_size(p), bh, G) in good
