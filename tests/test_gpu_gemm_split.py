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
                                   (321, 4096, 3072), (1800, 576, 256), (4096, 64, 512), (1024, 1152, 4096), (300, 3584, 512),
                                   (320, 4096, 1536)])
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


def _same_class(got, ref):
    """The infinities and NaNs of the float64 result, and its values elsewhere."""
    ref, got = ref.double(), got.double()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.where(torch.isinf(got), got.sign(), 0), torch.where(torch.isinf(ref), ref.sign(), 0))
    fin = torch.isfinite(ref)
    assert float((got - ref)[fin].norm() / ref[fin].norm()) < 1e-6


@pytest.mark.parametrize("half", [True, False])
def test_gemm_split_nonfinite(K, half):
    """Infinities and NaNs reach their own row and column only (fp32 values past fp16's range are
    infinities to the product)."""
    g = torch.Generator(device=DEV).manual_seed(9)
    m, n, k = 70, 80, 512
    a, w = torch.randn(m, k, generator=g, device=DEV), (torch.randn(n, k, generator=g, device=DEV) * 0.05).half()
    a[3, 100], a[20, 40], a[33, 511], a[64, 0], a[69, 300] = float("inf"), float("-inf"), float("nan"), 6e4, 7e4
    w[50, 7], w[51, 8] = float("inf"), float("nan")
    _same_class(K.gemm_f16(a.half() if half else a, w), a.half().double() @ w.double().T)


@pytest.mark.parametrize("m,ffn,k", [(70, 48, 512), (700, 4864, 512), (7937, 528, 128)])
def test_silu_nonfinite(K, m, ffn, k):
    """The SiLU products (the split, 256 x 256 tiles by columns and in rounds) with infinities and
    NaNs: the bits of the plain product and silu_mul, NaN where those are."""
    g = torch.Generator(device=DEV).manual_seed(m)
    a, w = torch.randn(m, k, generator=g, device=DEV).half(), (torch.randn(2 * ffn, k, generator=g, device=DEV) * 0.05).half()
    a[3, 100], a[20, 40], a[33, k - 1], a[64, 0], a[m - 1, 30] = float("inf"), float("-inf"), float("nan"), 6e4, -6e4
    got, ref = K.gemm_f16_silu(a, K.interleave_gate_up_f16(w), half=True), K.silu_mul(K.gemm_f16(a, w), ffn).half()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(got.nan_to_num(0.0, 1e4, -1e4), ref.nan_to_num(0.0, 1e4, -1e4))
