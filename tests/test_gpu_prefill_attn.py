"""The prefill attention on the fp32 matrix cores.

Tolerance: fp32 sums of up to 260 terms and the softmax's exponents, |score| * 2^-24 each with
scores up to ~20 here: 5e-6 relative in the 2-norm.
"""

import numpy as np
import pytest

from oracle import closed

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def K():
    from pico_hip import kernels
    return kernels


def err(got, ref):
    return float(np.linalg.norm(got.double().cpu().numpy() - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("L,pos0,nh,nkv,hd", [(1, 0, 14, 2, 64), (32, 0, 2, 2, 64), (33, 31, 14, 2, 64),
                                              (130, 5, 28, 4, 128), (257, 0, 4, 1, 128)])
def test_prefill_attn_matrix_cores(K, L, pos0, nh, nkv, hd):
    """The matrix-core kernel and the general kernel (taken for a V that is
    not 16-byte aligned) against float64."""
    rng = np.random.default_rng(L)
    q = (rng.standard_normal((L, nh, hd)) * 1.5).astype(np.float32)
    k, v = ((rng.standard_normal((nkv, pos0 + L + 3, hd)) * 1.5).astype(np.float32) for _ in range(2))
    ref = closed.causal_attention(q, k, v, pos0).reshape(L, nh * hd)
    qd, kd, vd = (torch.from_numpy(a).to(DEV) for a in (q, k, v))
    out = K.prefill_attn(qd, kd, vd, pos0=pos0)
    assert err(out, ref) < 5e-6
    odd = torch.empty(v.size + 1, device=DEV)[1:].view(v.shape).copy_(vd)
    assert err(K.prefill_attn(qd, kd, odd, pos0=pos0), ref) < 5e-6


def test_prefill_attn_later_nonfinite_values(K):
    """An infinity or a NaN in a later token's V row does not reach the queries before it."""
    g = torch.Generator(device=DEV).manual_seed(0)
    q, k, v = (torch.randn(s, generator=g, device=DEV) for s in ((50, 4, 64), (2, 50, 64), (2, 50, 64)))
    clean = K.prefill_attn(q, k, v)
    v[0, 20, 3], v[1, 40, 5], k[0, 45] = float("nan"), float("inf"), float("nan")
    got = K.prefill_attn(q, k, v)
    assert torch.allclose(got[:20], clean[:20], rtol=0, atol=2e-6)
    assert bool(torch.isnan(got[20:, 3]).all()) and bool(torch.isinf(got[40:, 2 * 64 + 5]).all())


@pytest.mark.parametrize("L,pos0,nh,nkv,hd", [(1, 0, 4, 2, 128), (33, 31, 14, 2, 64), (130, 5, 28, 4, 128)])
def test_prefill_attn_h16_holds_the_same_rows(K, L, pos0, nh, nkv, hd):
    g = torch.Generator(device=DEV).manual_seed(L)
    q, k, v = (torch.randn(s, generator=g, device=DEV) for s in ((L, nh, hd), (nkv, pos0 + L, hd), (nkv, pos0 + L, hd)))
    assert torch.equal(K.prefill_attn_h16(q, k, v, pos0=pos0), K.prefill_attn(q, k, v, pos0=pos0).half())
    odd = torch.empty(v.numel() + 1, device=DEV)[1:].view(v.shape).copy_(v)   # not 16-byte aligned
    assert torch.equal(K.prefill_attn_h16(q, k, odd, pos0=pos0), K.prefill_attn(q, k, odd, pos0=pos0).half())


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("form", ["fp32", "fp16", "x3"])
def test_prefill_attn_nan_keys_reach_the_rows_that_see_them(K, hd, form):
    """A NaN score makes its query's row NaN, also where the NaN keys are all that one of the
    merged parts sees (keys 32, 64 and 96 for the queries at their own position, whole key tiles
    for later ones); rows that see no NaN key keep their values."""
    from test_gpu_x3 import from_x3
    L, nh, nkv = 200, 4, 2
    g = torch.Generator(device=DEV).manual_seed(hd)
    q, k, v = (torch.randn(s, generator=g, device=DEV) for s in ((L, nh, hd), (nkv, L, hd), (nkv, L, hd)))

    def run(kk):
        if form == "fp32":
            return K.prefill_attn(q, kk, v)
        if form == "fp16":
            return K.prefill_attn_h16(q, kk, v).float()
        return from_x3(K.prefill_attn_x3(q, kk, v), L, nh * hd)

    clean = run(k).view(L, nkv, -1)
    for first, last in ((32, 33), (64, 65), (96, 97), (32, 64), (96, 128), (128, 160)):
        bad = k.clone()
        bad[1, first:last, hd // 2] = float("nan")     # one kv head: the other's rows stay
        got = run(bad).view(L, nkv, -1)
        assert torch.equal(got[:, 0], clean[:, 0])
        assert torch.equal(got[:first, 1], clean[:first, 1])
        assert bool(torch.isnan(got[first:, 1]).all()), (first, last)


def test_prefill_attn_operand_checks(K):
    """What the kernels would read or write past its end is refused: caches of another type, shape
    or order, queries of another type or head size."""
    q, k = torch.randn(5, 4, 64, device=DEV), torch.randn(2, 9, 64, device=DEV)
    bad = [(q, k.half(), k.half()), (q, k, k[:, :5].contiguous()), (q, k.transpose(0, 1).contiguous().transpose(0, 1), k),
           (q, k[..., :32].contiguous(), k[..., :32].contiguous())]
    for f in (K.prefill_attn_h16, K.prefill_attn_x3):
        for args in bad:
            with pytest.raises(ValueError):
                f(*args)
    with pytest.raises(ValueError):
        K.prefill_attn_h16(q.half(), k, k)


@pytest.mark.parametrize("L,pos0,nh,nkv,hd", [(1, 19, 14, 2, 64), (13, 0, 14, 2, 64), (20, 0, 28, 4, 128), (2, 18, 28, 4, 128),
                                              (21, 0, 14, 2, 64)])
def test_prefill_attn_few_keys(K, L, pos0, nh, nkv, hd):
    """Up to 20 keys the general kernel is the faster one: its bits (it is the one that takes a V
    that is not 16-byte aligned); past them the matrix cores."""
    g = torch.Generator(device=DEV).manual_seed(L)
    q, k, v = (torch.randn(s, generator=g, device=DEV) for s in ((L, nh, hd), (nkv, pos0 + L, hd), (nkv, pos0 + L, hd)))
    odd = torch.empty(v.numel() + 1, device=DEV)[1:].view(v.shape).copy_(v)
    assert torch.equal(K.prefill_attn(q, k, v, pos0=pos0), K.prefill_attn(q, k, odd, pos0=pos0)) == (pos0 + L <= 20)
