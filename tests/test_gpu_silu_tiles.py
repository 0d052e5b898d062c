"""The SiLU product of the prefill on 256 x 256 tiles from 512 rows on: the bits of the plain
product and silu_mul, which accumulate in the same order. Sizes: the first row count of the rule
and the one before it, ragged rows and columns, fewer column tiles than XCDs, tile counts that are
not a multiple of the XCDs, the shortest K, the rounds' grid from 32 row tiles on, and both sides of
the rule by K and tile count (the smaller tiles keep the short K, the few tiles and a nearly empty
second round)."""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("m,ffn,k", [(511, 1312, 128), (512, 1312, 128), (777, 4864, 896), (1000, 2064, 320),
                                     (1537, 4864, 128), (1601, 528, 192), (7937, 1040, 128),
                                     (512, 5120, 512), (512, 4864, 2048), (700, 4752, 256), (6100, 1040, 512),
                                     (2049, 1040, 1024), (1537, 4864, 896), (700, 2048, 896)])
def test_silu_tiles(m, ffn, k):
    from pico_hip import kernels as K
    g = torch.Generator(device=DEV).manual_seed(m + ffn)
    a = torch.randn(m, k, generator=g, device=DEV).half()
    w = (torch.randn(2 * ffn, k, generator=g, device=DEV) * 0.05).half()
    ref = K.silu_mul(K.gemm_f16(a, w), ffn).half()
    assert torch.equal(K.gemm_f16_silu(a, K.interleave_gate_up_f16(w), half=True), ref)
