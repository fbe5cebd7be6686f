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
