"""The embedding gather of four elements per thread, the row norm with the row in registers, and the
SiLU product with its fp16 roundings in one pass."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _err(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.fixture(scope="module")
def K():
    from pico_hip import kernels
    return kernels


# every format; rows shorter than a workgroup, a second column chunk with a remainder; an id count
# past the test's vocabulary
@pytest.mark.parametrize("name,hidden", [("Q5_0", 32), ("Q8_0", 896), ("Q8_0", 3584), ("Q4_K", 1280), ("Q6_K", 256),
                                         ("F16", 68), ("F32", 1028), ("F32", 66)])
def test_embed_gather_formats(K, name, hidden):
    from helpers import dequant_rows, dq, random_quant
    t = {"F32": 0, "F16": 1}.get(name)   # F32 and F16 rows need not be whole blocks
    rng = np.random.default_rng(hidden)
    if t is None:
        t = getattr(dq, name)
        raw = random_quant(t, 9, hidden, seed=hidden)
        ref = dequant_rows(t, raw, 9, hidden)
    else:
        w = rng.standard_normal((9, hidden)).astype(np.float16 if t else np.float32)
        raw, ref = w.tobytes(), w.astype(np.float32)
    ids = torch.tensor([0, 8, 3, 3, -1, 9, 5], device=DEV)
    out = K.embed_gather(K.RawTensor(torch.frombuffer(bytearray(raw), dtype=torch.uint8).to(DEV), t, (9, hidden)), ids).cpu().numpy()
    np.testing.assert_array_equal(out[[0, 1, 2, 3, 6]], ref[[0, 8, 3, 3, 5]])
    assert np.all(np.isnan(out[4:6]))


# ids on both sides of the rule between the two gathers (2^19 elements)
@pytest.mark.parametrize("name,hidden", [("Q5_0", 96), ("Q4_K", 256), ("Q6_K", 512), ("F16", 68)])
def test_embed_gather_many_ids(K, name, hidden):
    from helpers import dq, random_quant
    t = 1 if name == "F16" else getattr(dq, name)
    raw = np.random.default_rng(1).standard_normal((9, hidden)).astype(np.float16).tobytes() if t == 1 else \
        random_quant(t, 9, hidden, seed=hidden)
    tab = K.RawTensor(torch.frombuffer(bytearray(raw), dtype=torch.uint8).to(DEV), t, (9, hidden))
    rows = K.embed_gather(tab, torch.arange(9, device=DEV))
    for n in ((1 << 19) // hidden - 1, (1 << 19) // hidden + 3):
        ids = torch.randint(0, 9, (n,), device=DEV)
        assert torch.equal(K.embed_gather(tab, ids), rows[ids])


# one element, the ends of the register ranges (1024 and 4096 elements), remainders of 256
@pytest.mark.parametrize("n", [1, 255, 896, 1024, 1025, 3584, 4096, 4097])
@pytest.mark.parametrize("rows", [1, 5])
def test_rmsnorm_rows(K, n, rows):
    g = torch.Generator(device=DEV).manual_seed(n)
    x, w = torch.randn(rows, n, generator=g, device=DEV), torch.randn(n, generator=g, device=DEV)
    xd = x.double()
    ref = xd / torch.sqrt((xd * xd).mean(1, keepdim=True) + 1e-6) * w.double()
    # n fp32 additions over 256 partial sums, then four roundings: below 16 units in the last place
    y = K.rmsnorm(x, w, 1e-6)
    assert _err(y.double().cpu().numpy(), ref.cpu().numpy()) < 16 * 2.0 ** -24
    assert torch.equal(K.rmsnorm(x, w, 1e-6, half=True), y.half())


# the first row counts that take a wave per row, the ends of its register ranges, a last workgroup
# that is not full: the bits of the workgroup form (fewer rows)
@pytest.mark.parametrize("rows,n", [(4096, 1), (4099, 63), (4097, 512), (32768, 513), (32769, 1024)])
def test_rmsnorm_many_short_rows(K, rows, n):
    g = torch.Generator(device=DEV).manual_seed(n)
    x, w = torch.randn(rows, n, generator=g, device=DEV), torch.randn(n, generator=g, device=DEV)
    some = torch.cat([x[:40], x[-40:]])
    for half in (False, True):
        y = K.rmsnorm(x, w, 1e-6, half=half)
        assert torch.equal(torch.cat([y[:40], y[-40:]]), K.rmsnorm(some, w, 1e-6, half=half))


def test_rmsnorm_more_rows_than_one_grid_holds(K):
    """2^24 workgroups of 256 threads are more than one launch takes."""
    rows = (1 << 24) + 3
    x = torch.randn(rows, 2, device=DEV)
    w = torch.tensor([0.5, 2.0], device=DEV)
    y = K.rmsnorm(x, w, 1e-6)
    ref = x.double() / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-6) * w.double()
    assert float((y - ref).norm() / ref.norm()) < 16 * 2.0 ** -24


# whole quads and not (ffn % 4, a row stride % 4), both column orders; values past fp16's range
@pytest.mark.parametrize("L,ffn,il,pad", [(1, 16, True, 0), (37, 1040, True, 0), (5, 48, True, 3), (3, 50, False, 0),
                                          (9, 516, False, 4)])
def test_silu_mul_round(K, L, ffn, il, pad):
    g = torch.Generator(device=DEV).manual_seed(ffn)
    gu = torch.randn(L, 2 * ffn + pad, generator=g, device=DEV)[:, :2 * ffn]
    gu[0, :4] = torch.tensor([7e4, -7e4, 1e-8, -30.0], device=DEV)
    nat = gu.contiguous()
    if il:
        q = nat.view(L, -1, 2, 16)
        nat = torch.cat([q[:, :, 0].reshape(L, -1), q[:, :, 1].reshape(L, -1)], dim=1)
    ref = K.silu_mul(K.round_f16_(nat.clone()), ffn).half()
    assert torch.equal(K.silu_mul_round_h16(gu, ffn, interleaved=il).nan_to_num(1.0), ref.nan_to_num(1.0))


def test_silu_mul_round_row_strides(K):
    """The rows' own stride is used: rows that share memory are refused, as silu_mul refuses them
    (they were read as if they lay one behind another), one row of any stride is taken."""
    row = torch.randn(1, 64, device=DEV)
    for f in (K.silu_mul, K.silu_mul_round_h16):
        with pytest.raises(Exception, match="status 3"):
            f(row.expand(5, 64), 32)
    assert torch.equal(K.silu_mul_round_h16(row.expand(1, 64), 32), K.silu_mul_round_h16(row.clone(), 32))
    one = torch.as_strided(row, (1, 64), (1, 1))
    assert torch.equal(K.silu_mul_round_h16(one, 32), K.silu_mul_round_h16(row, 32))
