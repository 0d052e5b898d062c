"""The fp32-grade matrix-core prefill: x3 operands, products and the whole prefill.

Tolerances: fp32 sums of exact products, compared with float64. A sum of K terms added in chains
of at most K / 32 + 32 fp32 additions errs by about sqrt(K / 32 + 32) * 2^-24 of its own size
(3e-6 relative in the 2-norm is ten times what K = 4864 gives).
"""

import numpy as np
import pytest

from helpers import dequant_rows, quantized_normal, random_quant
from oracle import closed
from oracle import dequant as dq

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def K():
    from pico_hip import kernels
    return kernels


def qweight(K, t, raw, n, k):
    return K.pack_weight(torch.from_numpy(np.frombuffer(raw, np.uint8).copy()).to(DEV), t, n, k)


def err(got, ref):
    got = got.double().cpu().numpy() if isinstance(got, torch.Tensor) else got
    return float(np.linalg.norm(got - ref) / np.linalg.norm(ref))


def from_x3(x3, m, k):
    """The fp32 values of an x3 buffer: the sum of its three bf16 planes."""
    rt, kb = (m + 31) // 32, k // 32
    p = x3[:rt * kb * 6144].view(rt, kb, 2, 3, 2, 32, 16).contiguous().view(torch.bfloat16)  # half, plane, g, row
    return p.float().sum(3).permute(0, 4, 1, 2, 3, 5).reshape(rt * 32, k)[:m]


def x3_sums(x3, m, k):
    rt = (m + 31) // 32
    s = x3[rt * (k // 32) * 6144:].view(torch.float32).view(rt, k // 128, 32, 4)
    return s.permute(0, 2, 1, 3).reshape(rt * 32, k // 32)[:m]


@pytest.mark.parametrize("m,k", [(1, 32), (33, 128), (64, 96)])
def test_split_is_exact(K, m, k):
    # bf16's last bit is 2^-133, the third part's 2^-23 of the value: exact from 2^-110 on, and
    # short by less than 2^-133 below
    x = torch.randn(m, k, device=DEV) * torch.logspace(-30, 30, k, device=DEV)
    x[0, :3] = torch.tensor([torch.finfo(torch.float32).max, 0.0, -1.0])
    x3 = K.x3_split(x)
    back = from_x3(x3, m, k).double()
    assert bool(((back == x.double()) | ((x.abs() < 2.0 ** -110) & ((back - x.double()).abs() < 2.0 ** -133))).all())
    if k % 128 == 0:
        ref = x.double().view(m, k // 32, 32).sum(2)
        assert float(((x3_sums(x3, m, k) - ref).abs() / x.double().abs().view(m, -1, 32).sum(2)).max()) < 32 * 2.0 ** -24
    y = x.clone()
    y[0, 5], y[0, 6], y[0, 7] = float("inf"), float("-inf"), float("nan")
    back = from_x3(K.x3_split(y), m, k)
    assert torch.isinf(back[0, 5]) and back[0, 6] == float("-inf") and torch.isnan(back[0, 7])


def row_err(got, ref):
    """The largest relative error of a row (2-norm)."""
    got = got.double().cpu().numpy()
    return float((np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)).max())


# every tile rule: one and two column tiles per workgroup, shared decode; ragged rows and columns;
# the shortest K (one step per format), K shares without a step, and long ones
SHAPES = [(dq.Q5_0, 64, 32), (dq.Q5_0, 896, 900), (dq.Q8_0, 192, 130), (dq.Q8_0, 896, 3584), (dq.Q4_K, 256, 33),
          (dq.Q4_K, 4864, 896), (dq.Q6_K, 256, 40), (dq.Q6_K, 4864, 896), (dq.Q4_K, 512, 3584), (dq.Q6_K, 512, 3584)]


@pytest.mark.parametrize("m", [1, 32, 33, 277, 500])
@pytest.mark.parametrize("t,k,n", SHAPES)
def test_qgemm_x3(K, m, t, k, n):
    raw = quantized_normal(t, n, k, seed=n)
    w = qweight(K, t, raw, n, k)
    rng = np.random.default_rng(m)
    x = rng.standard_normal((m, k)).astype(np.float32)
    r = rng.standard_normal((m, n)).astype(np.float32)
    out = torch.from_numpy(r).to(DEV)
    K.qgemm_x3(K.x3_split(torch.from_numpy(x).to(DEV)), m, w, residual=out, out=out)  # in place
    ref = x.astype(np.float64) @ dequant_rows(t, raw, n, k).astype(np.float64).T + r
    assert err(out, ref) < 3e-6
    again = torch.from_numpy(r).to(DEV)
    K.qgemm_x3(K.x3_split(torch.from_numpy(x).to(DEV)), m, w, residual=again, out=again)
    assert torch.equal(out, again)


@pytest.mark.parametrize("m", [4, 400])
def test_qgemm_reads_the_weights_columns(K, m):
    """qgemm of rows wider than the matrix uses their first k columns, on the dot products (4 rows)
    and on the matrix cores (400 rows); rows that are shorter are refused on both."""
    t, n, k = dq.Q8_0, 256, 512
    raw = quantized_normal(t, n, k, seed=1)
    w = qweight(K, t, raw, n, k)
    x = torch.randn(m, k + 96, device=DEV)
    ref = x[:, :k].double().cpu().numpy() @ dequant_rows(t, raw, n, k).astype(np.float64).T
    assert err(K.qgemm(x, w), ref) < 3e-6
    assert err(K.qgemm(x[:, None], w), ref) < 3e-6     # rows of a 3-d tensor
    for bad in (torch.randn(m, k - 64, device=DEV), torch.randn(1, k, device=DEV).expand(m, k)):
        with pytest.raises(Exception, match="status 3"):
            K.qgemm(bad, w)


def test_qgemm_of_many_rows(K):
    """More rows than one conversion takes: the bits of the rows by themselves, in strided operands
    and with a residual, and a scratch that does not grow with the rows."""
    t, n, k, m = dq.Q8_0, 96, 512, 2 * 8192 + 70
    w = qweight(K, t, quantized_normal(t, n, k, seed=1), n, k)
    x = torch.randn(m, k + 4, device=DEV)[:, :k]
    res, bias = torch.randn(m, n + 1, device=DEV)[:, :n], torch.randn(n, device=DEV)
    out = torch.full((m, n + 2), 7.0, device=DEV)
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    K.qgemm(x, w, bias=bias, residual=res, out=out[:, :n])
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - base <= 8192 * k * 6 + 8192 * k // 8 + (2 << 20)
    assert bool((out[:, n:] == 7).all())
    for a, b in ((0, 500), (8000, 8500), (15900, m)):
        assert torch.equal(out[a:b, :n], K.qgemm(x[a:b], w, bias=bias, residual=res[a:b]))


@pytest.mark.parametrize("m", [1, 64, 65, 401])
@pytest.mark.parametrize("t,k,ffn", [(dq.Q5_0, 64, 96), (dq.Q8_0, 128, 128), (dq.Q4_K, 256, 8192), (dq.Q6_K, 512, 160)])
def test_qgemm_x3_silu(K, m, t, k, ffn):
    raw = quantized_normal(t, 2 * ffn, k, seed=ffn)
    w = qweight(K, t, raw, 2 * ffn, k)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    x3 = K.qgemm_x3_silu(K.x3_split(torch.from_numpy(x).to(DEV)), m, w)
    gu = x.astype(np.float64) @ dequant_rows(t, raw, 2 * ffn, k).astype(np.float64).T
    ref = closed.silu_mul(gu[:, :ffn], gu[:, ffn:])
    got = from_x3(x3, m, ffn)
    assert err(got, ref) < 3e-6
    if ffn % 128 == 0:
        sums = got.double().view(m, ffn // 32, 32).sum(2).cpu().numpy()
        assert err(x3_sums(x3, m, ffn), sums) < 1e-6


# the shared decode over several rounds of its double buffer and several flushes of its partial sums
# (every four sub-steps): the rows' K of the two model shapes, K shares of unequal length (Q5_0, 960),
# a ragged last pair of row tiles; four row tiles sharing it (from 8192 columns on)
@pytest.mark.parametrize("t,k,ffn,m", [(dq.Q5_0, 896, 160, 65), (dq.Q5_0, 896, 160, 277), (dq.Q5_0, 960, 96, 130),
                                       (dq.Q8_0, 896, 96, 277), (dq.Q4_K, 3584, 96, 65), (dq.Q4_K, 3584, 96, 277),
                                       (dq.Q6_K, 1536, 96, 65), (dq.Q6_K, 1536, 96, 277), (dq.Q5_0, 960, 8192, 401),
                                       (dq.Q4_K, 1280, 8192, 401)])
def test_qgemm_x3_silu_long_k(K, t, k, ffn, m):
    raw = random_quant(t, 2 * ffn, k, seed=ffn + k)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    x3 = K.qgemm_x3_silu(K.x3_split(torch.from_numpy(x).to(DEV)), m, qweight(K, t, raw, 2 * ffn, k))
    gu = x.astype(np.float64) @ dequant_rows(t, raw, 2 * ffn, k).astype(np.float64).T
    assert row_err(from_x3(x3, m, ffn), closed.silu_mul(gu[:, :ffn], gu[:, ffn:])) < 3e-6


# the same in the plain product (from 1536 tiles on)
@pytest.mark.parametrize("t,k", [(dq.Q5_0, 896), (dq.Q5_0, 960), (dq.Q8_0, 960), (dq.Q4_K, 1280), (dq.Q6_K, 1536)])
def test_qgemm_x3_shared_long_k(K, t, k):
    n, m = 3584, 449
    raw = random_quant(t, n, k, seed=k)
    x = np.random.default_rng(k).standard_normal((m, k)).astype(np.float32)
    got = K.qgemm_x3(K.x3_split(torch.from_numpy(x).to(DEV)), m, qweight(K, t, raw, n, k))
    assert row_err(got, x.astype(np.float64) @ dequant_rows(t, raw, n, k).astype(np.float64).T) < 3e-6


@pytest.mark.parametrize("t", [dq.Q5_0, dq.Q8_0, dq.Q4_K, dq.Q6_K])
@pytest.mark.parametrize("kind", ["normal", "one block", "one column", "even blocks", "odd blocks"])
def test_qgemm_x3_signed_error(K, t, kind):
    """Rows whose energy sits in one block or in blocks of one parity, where the alternating signs do
    not take the downward rounding of the matrix cores' sums out: the error stays that of fp32 sums
    row by row, and its mean is at most half a unit in the last place of each block's sum for each
    of the two additions at its full size (2 * 2^-24); with ordinary rows the mean is gone."""
    n, k, m = 896, 4864, 40
    raw = quantized_normal(t, n, k, seed=5)
    x = np.random.default_rng(6).standard_normal((m, k)).astype(np.float32)
    block = np.arange(k) // 32
    for r in range(m):
        big = {"normal": np.zeros(k, bool), "one block": block == 7 * r % (k // 32),
               "one column": np.arange(k) == 37 * r + 5, "even blocks": block % 2 == 0, "odd blocks": block % 2 == 1}[kind]
        x[r, big] *= 1000.0
    w = dequant_rows(t, raw, n, k).astype(np.float64)
    ref = x.astype(np.float64) @ w.T
    got = K.qgemm_x3(K.x3_split(torch.from_numpy(x).to(DEV)), m, qweight(K, t, raw, n, k))
    assert row_err(got, ref) < 1e-6
    d = (got.double().cpu().numpy() - ref).mean(axis=1)
    parts = np.abs(np.einsum("mbk,nbk->mnb", x.astype(np.float64).reshape(m, -1, 32), w.reshape(n, -1, 32), optimize=True))
    assert np.all(np.abs(d) <= 2 * 2.0 ** -24 * parts.sum(axis=2).mean(axis=1) + 4e-7 * np.abs(ref).mean(axis=1) / np.sqrt(n))
    if kind == "normal":    # 40 x 896 errors of about 1e-7 of |y|: their mean within 2e-9 of zero
        assert abs(float((d / np.abs(ref).mean(axis=1)).mean())) < 1e-8


EXTREMES = (float("inf"), float("-inf"), float("nan"), 3e38, -1e37)


def same_class(got, ref):
    """Finite where the float64 result is (as float32), with its values; else the same infinities
    and NaNs."""
    with np.errstate(over="ignore"):
        ref = np.asarray(ref, np.float64).astype(np.float32)
    got = got.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.where(np.isinf(got), np.sign(got), 0), np.where(np.isinf(ref), np.sign(ref), 0))
    fin = np.isfinite(ref)
    # a row with a huge element is that element times a weight: fp32 rounding of each value; the
    # other rows by their own size
    got, ref = np.where(fin, got, 0).astype(np.float64), np.where(fin, ref, 0).astype(np.float64)
    tol = 4e-6 * np.sqrt(np.mean(ref ** 2, axis=-1, keepdims=True))
    assert np.all(np.abs(got - ref) <= tol + 4e-6 * np.abs(ref))


def extreme_rows(m, k, rng):
    x = rng.standard_normal((m, k)).astype(np.float32)
    for i, v in enumerate(EXTREMES):
        x[(7 * i + 2) % m, (37 * i + 5) % k] = v
    return x


@pytest.mark.parametrize("t", [dq.Q5_0, dq.Q8_0, dq.Q4_K, dq.Q6_K])
@pytest.mark.parametrize("m,n,k", [(40, 96, 512), (200, 8320, 256)])
def test_qgemm_x3_nonfinite(K, t, m, n, k):
    """Infinities, NaNs and values near the end of fp32's range give what the fp32 product gives
    (one column tile per workgroup, and the shared decode), in their own rows only."""
    raw = quantized_normal(t, n, k, seed=n)
    w, x = qweight(K, t, raw, n, k), extreme_rows(m, k, np.random.default_rng(1))
    r = np.random.default_rng(2).standard_normal((m, n)).astype(np.float32)
    got = K.qgemm_x3(K.x3_split(torch.from_numpy(x).to(DEV)), m, w, residual=torch.from_numpy(r).to(DEV))
    with np.errstate(invalid="ignore"):
        same_class(got, x.astype(np.float64) @ dequant_rows(t, raw, n, k).astype(np.float64).T + r)


@pytest.mark.parametrize("t", [dq.Q5_0, dq.Q8_0, dq.Q4_K, dq.Q6_K])
@pytest.mark.parametrize("m", [40, 100])
def test_qgemm_x3_silu_and_qkv_nonfinite(K, t, m):
    k, ffn, nh, nkv, hd = 512, 96, 3, 1, 64
    x = extreme_rows(m, k, np.random.default_rng(3))
    x3 = K.x3_split(torch.from_numpy(x).to(DEV))
    raw = quantized_normal(t, 2 * ffn, k, seed=4)
    with np.errstate(all="ignore"):
        gu = x.astype(np.float64) @ dequant_rows(t, raw, 2 * ffn, k).astype(np.float64).T
        gu = gu.astype(np.float32).astype(np.float64)      # gate and up are fp32 values
        ref = closed.silu_mul(gu[:, :ffn], gu[:, ffn:])
    same_class(from_x3(K.qgemm_x3_silu(x3, m, qweight(K, t, raw, 2 * ffn, k)), m, ffn), ref)
    tv = {dq.Q5_0: dq.Q8_0, dq.Q8_0: dq.Q5_0, dq.Q4_K: dq.Q6_K, dq.Q6_K: dq.Q4_K}[t]
    types, rows = (t, t, tv), (nh * hd, nkv * hd, nkv * hd)
    raws = [quantized_normal(f, n, k, seed=i + n) for i, (f, n) in enumerate(zip(types, rows))]
    ws = [qweight(K, f, b, n, k) for f, b, n in zip(types, raws, rows)]
    one, zero = torch.ones(m, hd // 2, device=DEV), torch.zeros(m, hd // 2, device=DEV)
    kc, vc = (torch.zeros(nkv, m, hd, device=DEV) for _ in range(2))
    q = K.qkv_x3(x3, m, *ws, None, None, None, one, zero, kc, vc, nh)
    with np.errstate(all="ignore"):
        ref = [(x.astype(np.float64) @ dequant_rows(f, b, n, k).astype(np.float64).T).reshape(m, -1, hd)
               for f, b, n in zip(types, raws, rows)]
        turn = lambda a: np.concatenate([a[..., :hd // 2] - a[..., hd // 2:] * 0.0, a[..., :hd // 2] * 0.0 + a[..., hd // 2:]], -1)
        same_class(q, turn(ref[0]))
        same_class(kc.transpose(0, 1), turn(ref[1]))
        same_class(vc.transpose(0, 1), ref[2])


@pytest.mark.parametrize("m", [2, 32, 33, 277])
@pytest.mark.parametrize("tq,tv,nh,nkv,hd,k", [(dq.Q5_0, dq.Q8_0, 14, 2, 64, 896), (dq.Q5_0, dq.Q5_0, 3, 1, 64, 64),
                                               (dq.Q4_K, dq.Q6_K, 4, 2, 128, 512), (dq.Q6_K, dq.Q4_K, 2, 1, 192, 256)])
def test_qkv_x3(K, m, tq, tv, nh, nkv, hd, k):
    types, rows = (tq, tq, tv), (nh * hd, nkv * hd, nkv * hd)
    raws = [quantized_normal(t, n, k, seed=i + n) for i, (t, n) in enumerate(zip(types, rows))]
    ws = [qweight(K, t, raw, n, k) for t, raw, n in zip(types, raws, rows)]
    rng = np.random.default_rng(m)
    x = rng.standard_normal((m, k)).astype(np.float32)
    bs = [rng.standard_normal(n).astype(np.float32) for n in rows]
    ang = rng.standard_normal((m, hd // 2))
    cos, sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    pos0, cap = 3, m + 7
    dev = [torch.from_numpy(a).to(DEV) for a in (*bs, cos, sin)]
    kc, vc = (torch.full((nkv, cap, hd), 7.0, device=DEV) for _ in range(2))
    q = K.qkv_x3(K.x3_split(torch.from_numpy(x).to(DEV)), m, *ws, *dev, kc, vc, nh, pos0=pos0)
    ref = [(x.astype(np.float64) @ dequant_rows(t, raw, n, k).astype(np.float64).T + b).reshape(m, -1, hd)
           for t, raw, n, b in zip(types, raws, rows, bs)]
    rot = lambda a: np.concatenate([a[..., :hd // 2] * cos[:, None] - a[..., hd // 2:] * sin[:, None],
                                    a[..., :hd // 2] * sin[:, None] + a[..., hd // 2:] * cos[:, None]], -1)
    assert err(q, rot(ref[0])) < 3e-6
    assert err(kc[:, pos0:pos0 + m], rot(ref[1]).transpose(1, 0, 2)) < 3e-6
    assert err(vc[:, pos0:pos0 + m], ref[2].transpose(1, 0, 2)) < 3e-6
    for c in (kc, vc):
        assert bool((c[:, :pos0] == 7).all()) and bool((c[:, pos0 + m:] == 7).all())


def test_qkv_x3_operand_checks(K):
    """Caches, biases and outputs the kernel would read or write past are refused."""
    nh, nkv, hd, k, m = 2, 1, 64, 64, 3
    w = [qweight(K, dq.Q8_0, quantized_normal(dq.Q8_0, n, k, seed=n), n, k) for n in (nh * hd, nkv * hd, nkv * hd)]
    x3, rot = K.x3_split(torch.randn(m, k, device=DEV)), torch.randn(m, hd // 2, device=DEV)
    kc, b = torch.zeros(nkv, 8, hd, device=DEV), torch.zeros(hd, device=DEV)
    run = lambda kk=kc, vv=kc.clone(), bk=b, out=None: K.qkv_x3(x3, m, *w, None, bk, None, rot, rot, kk, vv, nh, out=out)
    run()
    for bad in (dict(kk=kc.half(), vv=kc.half()), dict(vv=kc[:, :4].contiguous()), dict(bk=b[:32]),
                dict(out=torch.empty(m, nh, hd, device=DEV, dtype=torch.float16)), dict(out=torch.empty(1, nh, hd, device=DEV))):
        with pytest.raises(ValueError):
            run(**bad)


@pytest.mark.parametrize("n,m", [(32, 5), (896, 33), (4864, 2)])
def test_x3_rmsnorm(K, n, m):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((m, n)).astype(np.float32)
    w = rng.standard_normal(n).astype(np.float32)
    x3 = K.x3_rmsnorm(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV), 1e-6)
    assert err(from_x3(x3, m, n), closed.rmsnorm(x, w, 1e-6)) < 1e-6


@pytest.mark.parametrize("L,pos0,nh,nkv,hd", [(33, 31, 14, 2, 64), (130, 5, 28, 4, 128)])
def test_prefill_attn_x3_holds_the_same_rows(K, L, pos0, nh, nkv, hd):
    g = torch.Generator(device=DEV).manual_seed(L)
    q, k, v = (torch.randn(s, generator=g, device=DEV) for s in ((L, nh, hd), (nkv, pos0 + L, hd), (nkv, pos0 + L, hd)))
    x3 = K.prefill_attn_x3(q, k, v, pos0=pos0)
    assert torch.equal(from_x3(x3, L, nh * hd), K.prefill_attn(q, k, v, pos0=pos0))
    ref = from_x3(x3, L, nh * hd).double().view(L, nh * hd // 32, 32).sum(2).cpu().numpy()
    assert err(x3_sums(x3, L, nh * hd), ref) < 1e-6


@pytest.fixture(scope="module")
def wide_model(model_dir):
    """Two layers of the 0.5B widths: the loops of the products at the depth of the real model."""
    from pico_hip import synth
    path = model_dir / "wide-2l.gguf"
    if not path.exists():
        synth.build(path, synth.tiny_arch(n_layers=2, hidden=896, n_head=14, n_kv=2, head_dim=64, ffn=4864, vocab=512), seed=9)
    return path


@pytest.mark.parametrize("L,pos0,model", [(2, 0, "tiny"), (33, 0, "tiny"), (100, 7, "tiny"), (65, 0, "wide"), (277, 30, "wide")])
def test_prefill_x3_matches_the_general_path(K, tiny_model, wide_model, L, pos0, model):
    """The whole fp32 prefill on the matrix cores against the per-operation path of models its
    products do not cover: logits and caches, from position 0 and behind a cached prefix."""
    from pico_hip.engine import Engine
    eng = Engine(tiny_model if model == "tiny" else wide_model)
    m = eng.model
    ids = torch.randint(0, eng.cfg.vocab_size, (pos0 + L,), device=DEV, generator=torch.Generator(device=DEV).manual_seed(L))
    pos = torch.arange(pos0 + L, device=DEV)
    outs = []
    for x3 in (True, False):
        cache = eng._empty_cache(pos0 + L + 3)
        assert m._prefill_x3_ok(cache)
        if not x3:
            m._prefill_x3_ok = lambda cache: False
        if pos0:
            m.forward(ids[:pos0], pos[:pos0], cache)
        outs.append([m.forward(ids[pos0:], pos[pos0:], cache)] + [t for kv in cache for t in kv])
    for a, b in zip(*outs):
        assert err(a, b.double().cpu().numpy()) < 1e-5
