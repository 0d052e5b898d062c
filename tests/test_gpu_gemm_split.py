"""The prefill GEMM of few output tiles (K divided over a workgroup's waves).

Tolerance: fp16 operands are exact in the comparison (the reference multiplies the rounded
values in float64); fp32 sums of K = 4864 terms err by about sqrt(K) * 2^-24 / 4 of their size,
1e-6 in the 2-norm with the four shares.
"""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def K():
    from pico_hip import kernels
    return kernels


# the smallest K; one row; ragged rows and columns (also N % 4); the largest tile counts (256 = 4 x
# 64, of long K 320 = 5 x 64) and the first past them, which keep the larger tiles; long K; a tile
# count that is not a multiple of the XCDs, and fewer column tiles than XCDs
@pytest.mark.parametrize("m,n,k", [(1, 64, 256), (65, 130, 256), (63, 33, 320), (320, 4096, 256), (321, 4096, 256),
                                   (1021, 896, 4864), (256, 4096, 256), (257, 4096, 320), (320, 4096, 3072),
                                   (321, 4096, 3072), (1800, 576, 256), (4096, 64, 512), (1024, 1152, 4096)])
@pytest.mark.parametrize("half", [True, False])
def test_gemm_split(K, m, n, k, half):
    g = torch.Generator(device=DEV).manual_seed(m + n)
    a, w = torch.randn(m, k, generator=g, device=DEV), (torch.randn(n, k, generator=g, device=DEV) * 0.05).half()
    bias, res = torch.randn(n, generator=g, device=DEV), torch.randn(m, n, generator=g, device=DEV)
    x = a.half() if half else a
    ref = a.half().double() @ w.double().T
    rel = lambda t, r: float((t.double() - r).norm() / r.norm())
    assert rel(K.gemm_f16(x, w), ref) < 1e-6
    assert rel(K.gemm_f16(x, w, bias=bias), ref + bias.double()) < 1e-6
    out = res.clone()
    K.gemm_f16(x, w, bias=bias, residual=out, out=out)   # in place
    assert rel(out, ref + bias.double() + res.double()) < 1e-6
    wide = torch.full((m, n + 3), 7.0, device=DEV)       # rows that are not 16-byte aligned
    K.gemm_f16(x, w, out=wide[:, 1:1 + n])
    assert rel(wide[:, 1:1 + n], ref) < 1e-6 and bool((wide[:, 0] == 7).all()) and bool((wide[:, 1 + n:] == 7).all())


@pytest.mark.parametrize("m,ffn,k", [(1, 16, 256), (65, 48, 320), (300, 1024, 256)])
def test_gemm_split_silu(K, m, ffn, k):
    """The SiLU form: the bits of the plain product and silu_mul, in each operand and output type."""
    g = torch.Generator(device=DEV).manual_seed(m + ffn)
    a, w = torch.randn(m, k, generator=g, device=DEV), (torch.randn(2 * ffn, k, generator=g, device=DEV) * 0.05).half()
    wil = K.interleave_gate_up_f16(w)
    ref = K.silu_mul(K.gemm_f16(a, w), ffn)
    assert torch.equal(K.gemm_f16_silu(a, wil), ref)
    assert torch.equal(K.gemm_f16_silu(a, wil, half=True), ref.half())
    assert torch.equal(K.gemm_f16_silu(a.half(), wil, half=True), ref.half())


@pytest.mark.parametrize("m,n,k", [(1024, 1152, 896), (1024, 4096, 256)])
def test_gemm_past_one_tile_per_cu(K, m, n, k):
    """Past 256 tiles k_gemm_h16_dl is the faster one (1024 x 1152 x 896 14.1 against 20.7 us): the
    bits of the same rows in a longer product, which it takes as well."""
    g = torch.Generator(device=DEV).manual_seed(m + n)
    a, w = torch.randn(2 * m, k, generator=g, device=DEV).half(), (torch.randn(n, k, generator=g, device=DEV) * 0.05).half()
    assert torch.equal(K.gemm_f16(a[:m], w), K.gemm_f16(a, w)[:m])
