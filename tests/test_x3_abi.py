"""Argument checks of the fp32-grade matrix-core prefill entries and the rule that sends qgemm to
them (no GPU)."""

import ctypes

import pytest

pytest.importorskip("torch")
P = ctypes.c_void_p


@pytest.fixture(scope="module")
def lib():
    from pico_hip._lib import lib
    return lib


def test_x3_argument_checks(lib):
    fake, odd = P(0x1000), P(0x1004)
    assert lib.pe_x3_bytes(33, 64) == 2 * 2 * 6144
    assert lib.pe_x3_bytes(1, 128) == 4 * 6144 + 128 * 4
    assert lib.pe_x3_bytes(0, 64) == lib.pe_x3_bytes(1, 48) == -3
    assert lib.pe_x3_split(fake, 60, 2, 64, fake, None) == 3
    assert lib.pe_x3_split(odd, 64, 2, 64, fake, None) == 4
    # a grid of 2^32 threads runs no workgroup: refused (64 threads a row, 512 a 32 x 64 tile)
    assert lib.pe_x3_split(fake, 64, 1 << 26, 64, fake, None) == 3
    assert lib.pe_x3_rmsnorm(fake, 64, fake, 1e-6, 1 << 26, 64, fake, None) == 3
    assert lib.pe_qgemm_x3(8, fake, 1 << 28, 64, fake, 32 * 64, None, None, 0, fake, 1 << 28, None) == 3
    assert lib.pe_qgemm_x3_silu(8, fake, 1 << 27, 64, fake, 32 * 128, fake, None) == 3
    assert lib.pe_x3_rmsnorm(fake, 64, None, 1e-6, 2, 64, fake, None) == 1
    for t, k, want in ((6, 64, 0), (6, 96, 3), (8, 896, 0), (12, 256, 0), (12, 128, 3), (14, 32768, 0),
                       (14, 33024, 3), (1, 256, 2), (0, 256, 2)):
        assert lib.pe_qgemm_x3_supported(t, 32, k) == want
    assert lib.pe_qgemm_x3_supported(8, 1 << 28, 64) == 0 and lib.pe_qgemm_x3_supported(8, (1 << 28) + 1, 64) == 3
    assert lib.pe_qgemm_x3(8, fake, 64, 896, fake, 0, None, None, 0, fake, 64, None) == 3
    assert lib.pe_qgemm_x3(8, fake, 64, 896, fake, 2, None, fake, 63, fake, 64, None) == 3
    assert lib.pe_qgemm_x3(8, odd, 64, 896, fake, 2, None, None, 0, fake, 64, None) == 4
    rows = lambda scratch, size, x=fake, xs=896, m=40: lib.pe_qgemm_x3_rows(8, fake, 64, 896, x, xs, m, None, None, 0, fake,
                                                                            64, scratch, size, None)
    assert rows(fake, lib.pe_x3_bytes(32, 896) - 1) == rows(fake, 0) == 6       # not one row tile
    assert rows(odd, 1 << 30) == 4 and rows(None, 1 << 30) == 1 and rows(fake, 1 << 30, m=0) == 3
    assert rows(fake, 1 << 30, xs=892) == 3 and rows(fake, 1 << 30, x=None) == 1
    assert lib.pe_qgemm_x3_silu(8, fake, 48, 896, fake, 2, fake, None) == 3     # ffn % 32
    assert lib.pe_qkv_x3_supported(6, 6, 8, 896, 14, 2, 64) == 0
    assert lib.pe_qkv_x3_supported(12, 12, 14, 3584, 28, 4, 128) == 0
    assert lib.pe_qkv_x3_supported(6, 8, 8, 896, 14, 2, 64) == 2                # q and k differ
    assert lib.pe_qkv_x3_supported(12, 12, 8, 256, 14, 2, 64) == 2              # block sizes differ
    assert lib.pe_qkv_x3_supported(6, 6, 6, 896, 14, 2, 32) == 3                # hd % 64
    assert lib.pe_prefill_attn_x3(fake, 896, fake, fake, 14, 2, 64, 77, 13, 70, 0.125, fake, None) == 3
    assert lib.pe_prefill_attn_x3(fake, 896, fake, odd, 14, 2, 64, 77, 13, 0, 0.125, fake, None) == 4
    assert lib.pe_prefill_attn_h16(fake, 896, fake, fake, 14, 2, 64, 77, 13, 0, 0.125, fake, 895, None) == 3
    assert lib.pe_prefill_attn_h16(fake, 896, fake, fake, 14, 2, 64, 77, 13, 0, 0.125, fake, 900, None) == 4
    assert lib.pe_prefill_attn_h16(fake, 896, fake, fake, 14, 2, 64, 77, 13, 0, 0.125, odd, 896, None) == 4


def test_qgemm_rule():
    from pico_hip import kernels as K
    assert not K._qgemm_x3_pays(0, 896, 896) and not K._qgemm_x3_pays(7, 896, 896)
    assert K._qgemm_x3_pays(8, 32, 64) and K._qgemm_x3_pays(3, 3584, 3584)
    assert not K._qgemm_x3_pays(2, 3584, 3584)


def test_qgemm_rule_of_long_rows():
    """Long rows go to the matrix cores by m n, not by the row count alone: a narrow matrix's dot
    products are 2 to 4 times faster there (128 x 4864, 8 rows 8.8 against 21 us)."""
    from pico_hip import kernels as K
    for m, n, k in ((8, 128, 4864), (16, 256, 18944), (8, 512, 3584), (4, 256, 32768), (2, 896, 18944), (1, 3584, 18944),
                    (64, 32, 8192)):
        assert not K._qgemm_x3_pays(m, n, k), (m, n, k)
    for m, n, k in ((8, 896, 4864), (2, 3584, 18944), (16, 512, 3584), (277, 128, 4864), (8, 128, 896), (3, 3584, 3584),
                    (1, 37888, 3584)):
        assert K._qgemm_x3_pays(m, n, k), (m, n, k)
    assert not K._qgemm_x3_pays(16, 512, 256, K.GGML_Q4_K) and K._qgemm_x3_pays(64, 512, 256, K.GGML_Q6_K)
    assert not K._qgemm_x3_pays(65535 * 8 + 1, 896, 896)    # pe_qgemm refuses those rows


def test_qgemm_rule_counts_the_second_launch():
    """Products of a few us stay on the one launch of the dot products, whatever the device time."""
    from pico_hip import kernels as K
    assert not any(K._saves_a_launch(m, n, k) for m, n, k in ((8, 32, 64), (8, 896, 896), (13, 128, 896), (8, 896, 4864),
                                                             (64, 128, 896)))
    assert all(K._saves_a_launch(m, n, k) for m, n, k in ((13, 896, 4864), (8, 9728, 896), (64, 896, 896), (2, 3584, 18944),
                                                         (277, 128, 896)))
