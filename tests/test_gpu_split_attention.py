"""The fused attention on bf16 parts (attn_fwd_kernel and its prepass), through MultiHeadAttention with
identity projections (exact in the split GEMM), so query = xq and key = value = xkv.

Bound per element, from the arithmetic, in units of 2^-24 and S = max over the keys of
sum |q||k| scale log2(e): a score (log2 units, relative to the reference maximum, which is at most S) is
off by 2 units of 2 S in each of hd / 16 accumulations of the large products, by 2 for adding the small
ones and taking off the maximum, 1 for the products left out, 3 for the scaled query: ds = (hd / 4 + 6)
units of S. A probability is off by a relative ds ln 2 + 2^-22 (the hardware exponential), numerator and
denominator each by that; the numerator rounds by 2 units of sum p |v| in at most 6 sums of 16 keys, the
denominator by Sk / 32 + 32, the quotient by 8:
|o - ref| <= (2 (ds ln 2 + 2^-22) + (12 Sk / 16 + Sk / 32 + 40) 2^-24) sum p |v|.
"""
import numpy as np
import pytest

from metalaudio_amd import nn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return nn.AudioDevice(0)


def run(dev, heads, xq, xkv):
    m = nn.MultiHeadAttention(dev, xq.shape[-1], heads)
    s = nn.Stream(dev)
    out = nn.Tensor(dev, xq.shape)
    dev.set_kernel_timing(True)
    dev.reset_kernel_timing()
    m.forward_cross(nn.Tensor.from_numpy(dev, xq), nn.Tensor.from_numpy(dev, xkv), out, s)
    s.sync(20000)
    parts = dev.kernel_timing("attn_parts")[0]
    dev.set_kernel_timing(False)
    return out.to_numpy(), parts


def check(y, xq, xkv, heads, rows):
    B, Sq, E = xq.shape
    hd, Sk = E // heads, xkv.shape[1]
    scale = 1 / np.sqrt(hd)
    for b in range(B):
        for h in range(heads):
            c = slice(h * hd, (h + 1) * hd)
            q, k = xq[b, rows][:, c].astype(np.float64), xkv[b][:, c].astype(np.float64)
            s = q @ k.T * scale
            p = np.exp(s - s.max(1, keepdims=True))
            p /= p.sum(1, keepdims=True)
            ds = (hd / 4 + 6) * 2.0 ** -24 * (np.abs(q) @ np.abs(k).T).max(1) * scale * 1.4427
            rel = 2 * (ds * np.log(2) + 2.0 ** -22) + (12 * Sk / 16 + Sk / 32 + 40) * 2.0 ** -24
            err = np.abs(y[b, rows][:, c] - p @ k)
            assert np.all(err <= rel[:, None] * (p @ np.abs(k))), (b, h, err.max())


# one block and many, ragged last keys and queries, every key-split count, both head dims
CASES = [(1, 8, 48, 1344, 1344), (4, 8, 48, 260, 509), (1, 8, 48, 2689, 333), (2, 8, 64, 777, 1501),
         (16, 8, 64, 256, 97), (1, 8, 64, 3000, 131), (4, 8, 48, 1027, 2050)]


@pytest.mark.parametrize("B,H,hd,Sq,Sk", CASES)
def test_parts_attention_error_bound(dev, B, H, hd, Sq, Sk):
    print(f"split attention {B, H, hd, Sq, Sk}", flush=True)
    r = np.random.default_rng(Sq + Sk)
    xq = r.standard_normal((B, Sq, H * hd)).astype(np.float32)
    xkv = (1.5 * r.standard_normal((B, Sk, H * hd))).astype(np.float32)
    y, parts = run(dev, H, xq, xkv)
    assert parts == 1
    check(y, xq, xkv, H, np.arange(0, Sq, max(1, Sq // 300)))


# 256 * Sk * 384 >= 2e8 from Sk = 2035 on
@pytest.mark.parametrize("Sq,Sk,parts", [(255, 4000, 0), (256, 2034, 0), (256, 2035, 1)])
def test_small_calls_stay_on_fp32_products(dev, Sq, Sk, parts):
    print(f"attention form {Sq, Sk}", flush=True)
    r = np.random.default_rng(Sq)
    xq = r.standard_normal((1, Sq, 384)).astype(np.float32)
    xkv = r.standard_normal((1, Sk, 384)).astype(np.float32)
    y, got = run(dev, 8, xq, xkv)
    assert got == parts
    check(y, xq, xkv, 8, np.arange(Sq))


def test_nan_query_leaves_the_others(dev):
    """A query row of NaN gives a row of NaN; the other queries of its wave, recomputed with fp32 products
    (scores of hd / 2 roundings, sums of Sk / 2), stay within the bound above, which covers those."""
    print("split attention NaN row", flush=True)
    r = np.random.default_rng(3)
    xq = r.standard_normal((1, 700, 384)).astype(np.float32)
    xkv = r.standard_normal((1, 900, 384)).astype(np.float32)
    xq[0, 37] = np.nan
    y, parts = run(dev, 8, xq, xkv)
    assert parts == 1 and np.all(np.isnan(y[0, 37]))
    check(y, xq, xkv, 8, np.array([i for i in range(700) if i != 37]))


@pytest.mark.parametrize("B,H,hd,Sq,Sk", [(1, 8, 48, 700, 900), (1, 8, 64, 700, 900),
                                          (1, 8, 48, 100, 200), (1, 4, 64, 60, 130)])
def test_low_scores_in_the_first_keys(dev, B, H, hd, Sq, Sk):
    """Finite scores far below -128 (log2 units) for the first 64 keys, or for every key: the result is
    the softmax's and takes no longer than ordinary scores (computed again in fp32 it would)."""
    print(f"split attention low scores {B, H, hd, Sq, Sk}", flush=True)
    r = np.random.default_rng(hd + Sq)
    xq = r.standard_normal((B, Sq, H * hd)).astype(np.float32)
    xkv = r.standard_normal((B, Sk, H * hd)).astype(np.float32)
    ordinary = min(timed(dev, H, xq, xkv)[1] for _ in range(3))
    u = r.standard_normal((H, hd))
    u = (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32).reshape(-1)
    xq[:, ::3] += 40 * u      # against the first keys: -40 * 40 * scale, about -230 or -200
    xkv[:, :64] -= 40 * u
    xq[:, 1::3] += 40 * u
    for shift in (0, 40):
        xkv[:, 64:] -= shift * u
        runs = [timed(dev, H, xq, xkv) for _ in range(3)]
        y = runs[0][0]
        assert np.all(np.isfinite(y))
        check(y, xq, xkv, H, np.arange(0, Sq, max(1, Sq // 300)))
        assert min(t for _, t in runs) < 3 * ordinary


def timed(dev, heads, xq, xkv):
    m = nn.MultiHeadAttention(dev, xq.shape[-1], heads)
    s = nn.Stream(dev)
    out = nn.Tensor(dev, xq.shape)
    q, kv = nn.Tensor.from_numpy(dev, xq), nn.Tensor.from_numpy(dev, xkv)
    m.forward_cross(q, kv, out, s)
    s.sync(20000)
    dev.set_kernel_timing(True)
    dev.reset_kernel_timing()
    m.forward_cross(q, kv, out, s)
    s.sync(20000)
    ms = dev.kernel_timing("attn_fwd")[1]
    dev.set_kernel_timing(False)
    return out.to_numpy(), ms


@pytest.mark.parametrize("hd", [48, 64])
def test_many_small_probabilities_beside_a_large_one(dev, hd):
    """One key's probability is 1, a thousand others are just above half of its last bit: added one by
    one onto a running sum each would count as a whole one. All values are 1, so the result is the
    numerator's sum of probabilities over the denominator's. In units of 2^-24: the denominator
    rounds by 1 a block of keys and by 32 within the first, the numerator by at most 2 in each of 3 sums
    of 16 keys, and the last quotient by 3."""
    print(f"split attention many small probabilities hd{hd}", flush=True)
    B, H, Sq, Sk = 8, 8, 640, 1024  # enough query blocks that the keys are not split
    E = H * hd
    m = nn.MultiHeadAttention(dev, E, H)
    eye = np.eye(E, dtype=np.float32)
    m.load_weights_named("in_proj_weight", np.concatenate([eye, eye, 0 * eye]))
    m.load_weights_named("in_proj_bias", np.repeat(np.float32([0, 0, 1]), E))
    xq = np.zeros((B, Sq, E), np.float32)
    xkv = np.zeros((B, Sk, E), np.float32)
    xq[:, :, ::hd] = 1
    xkv[:, 0, ::hd] = 23.9 * np.log(2) * np.sqrt(hd)
    out, s = nn.Tensor(dev, xq.shape), nn.Stream(dev)
    m.forward_cross(nn.Tensor.from_numpy(dev, xq), nn.Tensor.from_numpy(dev, xkv), out, s)
    s.sync(20000)
    units = Sk / 32 + 32 + 2 * 3 * Sk / 16 + 3
    assert np.abs(out.to_numpy() - 1).max() <= units * 2.0 ** -24


# 2-norm of the error of the same inputs with fp32 products (v_mfma_f32_16x16x4_f32), head dim 48 and 64
FP32 = {"normal": (1.96e-7, 2.16e-7), "peaked": (6.14e-7, 7.11e-7), "one dim": (2.00e-7, 1.99e-7),
        "few keys": (5.29e-7, 5.76e-7)}


@pytest.mark.parametrize("kind", FP32)
@pytest.mark.parametrize("hd", [48, 64])
def test_no_further_off_than_fp32_products(dev, hd, kind):
    print(f"split attention against fp32 products {kind} hd{hd}", flush=True)
    r = np.random.default_rng(5)
    H, Sq, Sk = 8, 900, 1100
    xq, xkv = r.standard_normal((1, Sq, H * hd)), r.standard_normal((1, Sk, H * hd))
    if kind == "peaked":
        xq, xkv = 3 * xq, 2 * xkv
    elif kind == "one dim":  # scores of a single product
        one = np.arange(hd) == r.integers(0, hd, (1, Sq, H, 1))
        xq = xq * (6 * one).reshape(xq.shape)
    elif kind == "few keys":
        xkv = xkv * np.where(np.arange(Sk) < 50, 4, 0.01)[:, None]
    xq, xkv = xq.astype(np.float32), xkv.astype(np.float32)
    y, parts = run(dev, H, xq, xkv)
    assert parts == 1
    q, k = (a[0].reshape(-1, H, hd).transpose(1, 0, 2).astype(np.float64) for a in (xq, xkv))
    s = q @ k.transpose(0, 2, 1) / np.sqrt(hd)
    p = np.exp(s - s.max(2, keepdims=True))
    ref = ((p / p.sum(2, keepdims=True)) @ k).transpose(1, 0, 2).reshape(Sq, H * hd)
    assert np.linalg.norm(y[0] - ref) <= FP32[kind][hd == 64] * np.linalg.norm(ref)


def test_tiny_values(dev):
    """Values whose low parts lie below bf16's range: computed again with fp32 products (scores near 0, sums
    of Sk / 2), within the bound above."""
    print("split attention tiny values", flush=True)
    r = np.random.default_rng(18)
    xq = r.standard_normal((1, 700, 384)).astype(np.float32)
    xkv = np.ldexp(r.standard_normal((1, 900, 384)), -118).astype(np.float32)
    y, parts = run(dev, 8, xq, xkv)
    assert parts == 1
    check(y, xq, xkv, 8, np.arange(0, 700, 7))


@pytest.mark.parametrize("hd", [48, 64])
def test_nan_key(dev, hd):
    """A key that is not a number (in every head, once projected) makes every query of its batch one and no
    other, in a time that stays within reach (one query after another on the vector units it was 150
    times an ordinary call's)."""
    print(f"split attention NaN key hd{hd}", flush=True)
    r = np.random.default_rng(21)
    H, Sq, Sk = 8, 1300, 1000
    xq = r.standard_normal((2, Sq, H * hd)).astype(np.float32)
    xkv = r.standard_normal((2, Sk, H * hd)).astype(np.float32)
    ordinary = min(timed(dev, H, xq, xkv)[1] for _ in range(3))
    xkv[1, 700, 3] = np.nan
    runs = [timed(dev, H, xq, xkv) for _ in range(3)]
    y = runs[0][0]
    assert np.all(np.isnan(y[1]))
    check(y[:1], xq[:1], xkv[:1], H, np.arange(0, Sq, 7))
    assert min(t for _, t in runs) < 10 * ordinary
